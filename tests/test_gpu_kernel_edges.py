"""The kernels at the sizes where their layouts change: tile edges of the drafting search, windows and histories around
the prefetched part and its 16-byte blocks, rows with many segment lists, the softcap where it saturates. Against the
CPU oracle, bit-exact (whole numbers) as in test_gpu_parity.py."""
import os
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))

from ferro_amd import workloads as W  # noqa: E402
from oracle import oracle as O  # noqa: E402
import ferro_amd as F  # noqa: E402
from parity_util import bf16_valued, compare, oracle_decode_loop  # noqa: E402

NT = min(16, os.cpu_count() or 1)


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    yield
    torch.cuda.synchronize()


def csr(hists):
    off = np.concatenate([[0], np.cumsum([len(h) for h in hists])]).astype(np.int64)
    return np.concatenate([np.asarray(h, np.int32) for h in hists] + [np.zeros(0, np.int32)]), off


def check(x, p, hists, u, kcap=64):
    hist, off = csr(hists)
    out = F.sample_batch(torch.from_numpy(x).cuda(), p, u, hist=hist, hist_off=off, kcap=kcap)
    torch.cuda.synchronize()
    g = {k: v.cpu().numpy() for k, v in out.items() if v is not None and not k.startswith("_")}
    o = O.sample_batch(x, hist, off, p, u, kcap=kcap, nthreads=NT)
    nb = compare(g, o, p, u, kcap)
    assert F.device_error() == 0
    return nb


@pytest.mark.parametrize("L", [1, 2, 4, 5, 63, 1023, 16383, 16384, 16385, 16388, 40000])
def test_lookup_draft_tile_edges(L):
    """The only match (of 4, 3, 2 or 1 tokens) at the history's start, at a tile's edge and right before the end."""
    rng = np.random.default_rng(L)
    hists, min_n, E = [], [], 3
    for n in (4, 3, 2, 1):
        for at in (0, 1, L - 16384 - 2, L - 16384, L - n - 1, L // 2):
            h = rng.integers(1000, 1 << 20, L).astype(np.int32)        # no chance matches of two tokens
            if 0 <= at and at + n < L:
                h[at:at + n] = h[L - n:]
                if at % 3 == 1 and at + n < L - n:
                    h[at + n] = E                                      # a match directly before eos is passed over
            hists.append(h)
            min_n.append(int(rng.integers(0, n + 1)))
    hist, off = csr(hists)
    draft, nd = F.lookup_draft(hist, off, 70, min_n=np.asarray(min_n, np.int32), eos_id=E, draft_ld=70)
    draft, nd = draft.cpu().numpy(), nd.cpu().numpy()
    for s, h in enumerate(hists):
        want = O.lookup_draft(h, 70, eos=E, min_n=min_n[s])
        assert nd[s] == len(want), (L, s)
        np.testing.assert_array_equal(draft[s, :nd[s]], want)
