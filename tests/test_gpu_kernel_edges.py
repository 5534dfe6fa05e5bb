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


@pytest.mark.parametrize("L", [16385, 16386, 16387, 16388, 32769, 32771])
def test_lookup_draft_before_the_history(L):
    """A history's first ids are not preceded by anything: id 0 (what a tile holds there) does not complete a match.
    Histories that end in 0s and their own first ids; a genuine shorter match elsewhere stays the one found."""
    rng = np.random.default_rng(L)
    hists, min_n = [], []
    for n in (1, 2, 3, 4):
        for lead in (0, 1, 2, 3):
            h = rng.integers(1000, 1 << 20, L).astype(np.int32)
            h[L - 4:] = 0
            if lead:
                h[L - lead:] = h[:lead]
            if n == 2:
                h[L // 2:L // 2 + 2] = h[L - 2:]
            hists.append(h)
            min_n.append(n)
    hist, off = csr(hists)
    draft, nd = F.lookup_draft(hist, off, 20, min_n=np.asarray(min_n, np.int32), eos_id=3, draft_ld=20)
    draft, nd = draft.cpu().numpy(), nd.cpu().numpy()
    for s, h in enumerate(hists):
        want = O.lookup_draft(h, 20, eos=3, min_n=min_n[s])
        assert nd[s] == len(want), (L, s)
        np.testing.assert_array_equal(draft[s, :nd[s]], want)


@pytest.mark.parametrize("H,V", [(511, 65536), (512, 65536), (513, 65536), (515, 262144), (516 + 8192, 262144),
                                 (517 + 8192 + 2048 + 3, 262144), (20011, 100004)])
def test_long_windows_and_history_copies(H, V):
    """Decode steps whose histories end before, at and after the prefetched ids, at every offset from a 16-byte
    boundary, and shares of a row's copy longer than the prefetched part."""
    rng = np.random.default_rng(H)
    S = 5
    p = W.make_params(S, temperature=0.7, top_k=50, repetition_penalty=1.3)
    p["repeat_last_n"][1] = H - 3
    p["penalty_from"][2] = 5
    p["softcap"][3] = 30.0
    hist0 = [list(W.zipf_ids(rng, V, H + s)) for s in range(S)]
    rows = [W.mixture_logits(rng, S, V) for _ in range(2)]
    seeds = list(range(1, S + 1))
    want, want_hist, want_off = oracle_decode_loop(rows, p, seeds, hist0)
    d = F.DeviceRng(np.asarray(seeds, np.uint64))
    hist, off = (torch.from_numpy(a).cuda() for a in csr(hist0))
    for k, x in enumerate(rows):
        tok, _, hist, off = F.decode_step(torch.from_numpy(x).cuda(), p, d, hist=hist, hist_off=off)
        np.testing.assert_array_equal(tok.cpu().numpy(), want[k])
    np.testing.assert_array_equal(off.cpu().numpy(), want_off)
    np.testing.assert_array_equal(hist[:int(off[-1])].cpu().numpy(), want_hist)
    assert F.device_error() == 0


@pytest.mark.parametrize("V,k", [(65537, 64), (65537, 1 + 16), (262144, 64), (262144, 5), (262144, 16), (150000, 40)])
def test_rows_with_many_segment_lists(V, k):
    """17 to 64 lists per row: even rows, every top candidate in one segment (its list alone holds them: past its
    prefetched head), one candidate per segment, ties across segments, fewer candidates than k."""
    rng = np.random.default_rng(V + k)
    x = (rng.standard_normal((6, V)) * 2).astype(np.float32)
    x[1, 4096:4096 + 200] += 30.0
    x[2, ::4096] += 30.0
    x[3] = bf16_valued(x[3])
    x[4, :] = 1.0
    x[5, :] = np.nan
    x[5, rng.choice(V, 7, replace=False)] = 2.0
    p = W.make_params(6, temperature=0.8, top_k=k, top_p=0.97, repetition_penalty=1.0)
    check(x, p, [[]] * 6, rng.random(6))


@pytest.mark.parametrize("cap,scale", [(30.0, 1.0), (30.0, 40.0), (0.5, 1.0), (30.0, 300.0)])
def test_softcap_where_it_saturates(cap, scale):
    """Capped rows from unclipped to wholly saturated (every top logit caps to the same value: ties by id), with and
    without a repetition penalty above and below 1."""
    rng = np.random.default_rng(int(cap * 10 + scale))
    V = 70000
    x = (rng.standard_normal((6, V)) * scale).astype(np.float32)
    x[0, 5] = np.inf
    x[1, 6] = -np.inf
    x[2, 7] = np.nan
    x[3] = np.abs(x[3]) + np.float32(20 * cap)             # saturated everywhere
    p = W.make_params(6, temperature=0.9, top_k=40, repetition_penalty=1.2)
    p["softcap"] = cap
    p["repetition_penalty"][4] = 0.8
    p["repetition_penalty"][5] = 1.0
    check(x, p, [list(W.zipf_ids(rng, V, 900)) for _ in range(6)], rng.random(6))


@pytest.mark.parametrize("cap", [1.0, 30.0, 0.375])
def test_softcap_never_decreases(cap):
    """Over every float from -inf to inf: bounds taken over raw logits hold for the capped ones."""
    import ctypes
    from ferro_amd._lib import lib
    chunk = 1 << 27
    out = torch.empty(chunk, dtype=torch.float32, device="cuda")
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    last = None
    for first in range(-0x7F800000, 0x7F800001, chunk):              # ascending floats: below 0 by their magnitude's bits
        i = torch.arange(first, min(first + chunk, 0x7F800001), dtype=torch.int64, device="cuda")
        x = torch.where(i < 0, -i, i).to(torch.int32).view(torch.float32)
        x = torch.where(i < 0, -x, x).contiguous()
        n = x.numel()
        assert lib().fs_softcap_batch(ctypes.c_void_p(x.data_ptr()), ctypes.c_void_p(out.data_ptr()), n,
                                      ctypes.c_float(cap), st) == 0
        y = out[:n]
        assert bool((y[1:] >= y[:-1]).all()) and (last is None or bool(y[0] >= last))
        last = y[-1].clone()


@pytest.mark.parametrize("V,k", [(5, 0), (40, 0), (64, 0), (65, 40), (320, 64), (800, 64), (2080, 50)])
@pytest.mark.parametrize("cap", [0.5, 30.0])
def test_softcap_and_penalties_on_short_rows(V, k, cap):
    """Rows too short for a bound from their lane maxima (every logit is then a candidate): penalised logits below -cap
    are candidates too. Windows of one id, of most and of all ids; -inf and NaN among the logits."""
    rng = np.random.default_rng(V)
    x = (rng.standard_normal((6, V)) * (2 if cap < 1 else 40)).astype(np.float32)
    x[4, rng.choice(V, V // 2, replace=False)] = -np.inf
    x[5, rng.choice(V, V // 2, replace=False)] = np.nan
    p = W.make_params(6, temperature=0.9, top_k=k, repetition_penalty=1.2)
    p["softcap"] = cap
    p["repetition_penalty"][3] = 2.0
    p["top_p"][1] = 0.9
    hists = [[int(x[0].argmin())], list(rng.permutation(V)[:V * 3 // 4]), *[list(range(V))] * 4]
    check(x, p, hists, np.array([0.999, 0.6, 0.999, 0.5, 0.9, 0.7]))


def mid_params(B, k, **kw):
    p = W.make_params(B, temperature=0.9, top_k=k, top_p=0.97, repetition_penalty=1.0)
    for f, v in kw.items():
        p[f] = v
    return p


@pytest.mark.parametrize("B,V,k", [(1, 4096, 65), (3, 33000, 1000), (2, 65537, 2048), (9, 100003, 66), (2, 262144, 2048),
                                   (70, 65536, 300), (33, 262144, 257)])
def test_mid_k_rows(B, V, k):
    """k past the small-k kernel's 64 on every segment size: heavy tails, bf16 values (ties at the k-th), every top
    logit in one segment, a masked vocabulary (fewer finite logits than k), an all-equal row, a row without a number."""
    rng = np.random.default_rng(V + k)
    x = W.mixture_logits(rng, B, V)
    if B > 1:
        x[1] = bf16_valued(x[1])
        x[B - 1, V // 3:V // 3 + 900] += 40.0
    if B > 2:
        m = np.full(V, -np.inf, np.float32)
        at = rng.choice(V, min(50, k // 2), replace=False)
        m[at] = x[2, at]
        x[2] = m
    if B > 8:
        x[3, :] = 2.5
        x[4, :] = np.nan
        x[5, rng.choice(V, V // 2, replace=False)] = np.nan
        x[6, 7] = np.inf
        x[7] = np.round(x[7])                        # thousands of equal logits at the bound
    check(x, mid_params(B, k), [[]] * B, rng.random(B), kcap=2048)


@pytest.mark.parametrize("V,B,H", [(100003, 6, 3000), (262144, 66, 2500), (70000, 4, 1), (70000, 4, 1025), (262144, 65, 9)])
def test_mid_k_penalties(V, B, H):
    """Every penalty mix, raising ones too; windows past the prefetched ids and histories whose distinct ids of one
    segment leave LDS for the spill list; every fourth row greedy, every fifth capped."""
    rng = np.random.default_rng(V + H)
    x = W.mixture_logits(rng, B, V)
    p = mid_params(B, 200, repetition_penalty=rng.choice([0.7, 1.0, 1.3], B), frequency_penalty=rng.choice([-0.2, 0.0, 0.3], B),
                   presence_penalty=rng.choice([0.0, 0.4], B))
    p["frequency_penalty"][0] = 0.1                  # at least one row past the small-k kernel
    p["temperature"][3::4] = 0.0
    p["softcap"][4::5] = 30.0
    p["repeat_last_n"][2::7] = max(1, H // 2)
    hists = [list(W.zipf_ids(rng, V, H)) if b % 3 else list(rng.integers(0, V, H)) for b in range(B)]
    hists[1] = list(rng.permutation(16384)[:H]) if H <= 16384 else hists[1]     # one segment's ids alone
    check(x, p, hists, rng.random(B), kcap=256)


@pytest.mark.parametrize("V,k", [(320, 10), (2080, 65), (4100, 100)])
@pytest.mark.parametrize("cap", [0.5, 30.0])
def test_mid_k_softcap_and_penalties_without_a_bound(V, k, cap):
    """Windows that hold every id (no logit is left to bound the row) or most, with penalties that take logits below
    -cap: they stay candidates. -inf and NaN among the logits."""
    rng = np.random.default_rng(V)
    x = (rng.standard_normal((6, V)) * (2 if cap < 1 else 40)).astype(np.float32)
    x[4, rng.choice(V, V // 2, replace=False)] = -np.inf
    x[5, rng.choice(V, V // 2, replace=False)] = np.nan
    p = mid_params(6, k, repetition_penalty=1.2, frequency_penalty=2.0)
    p["softcap"] = cap
    p["repetition_penalty"][3] = 2.0
    p["frequency_penalty"][3] = 0.0
    hists = [list(range(V)) * 20, list(rng.permutation(V)[:V * 3 // 4]) * 3, *[list(range(V))] * 4]
    check(x, p, hists, rng.random(6), kcap=k)


@pytest.mark.parametrize("k", [200, 1500, 2048])
def test_mid_k_lists_of_equal_logits(k):
    """Candidate lists of a few values: whole numbers, two neighbouring floats below one far larger logit (both fall in one
    bin of the sort, their ids in one bin of the next), equal logits at neighbouring ids."""
    rng = np.random.default_rng(k)
    B, V = 5, 100000
    x = np.full((B, V), -5.0, np.float32) + rng.random((B, V)).astype(np.float32)
    x[0] = np.round(rng.standard_normal(V) * 2)
    at = rng.permutation(V)
    x[1, at[:1100]] = 3.0
    x[1, at[1100:2100]] = np.nextafter(np.float32(3.0), np.float32(4.0))
    x[1, 17] = 1e6
    x[2, 5000:6000] = 2.0
    x[2, 90000:90700] = 2.0
    x[2, at[:90]] = 2.5
    x[3, at[:2400]] = bf16_valued(x[3, at[:2400]] * 0.01 + 6)
    x[4, at[:700]] = 1.0
    x[4, at[700:1500]] = 2.0
    x[4, at[1500:2300]] = 3.0
    check(x, mid_params(B, k, temperature=2.0), [[]] * B, rng.random(B), kcap=2048)


@pytest.mark.parametrize("B,V,k", [(9, 4100, 100), (9, 33000, 1000), (9, 100003, 70), (18, 100003, 2048), (9, 262144, 300),
                                   (66, 262144, 600)])
@pytest.mark.parametrize("cap", [0.0, 0.5, 30.0])
def test_mid_k_bounds_of_equal_logits(B, V, k, cap):
    """Rows whose k-th logit is one value of many: masks, coarse logits, one value; every third with penalties on tied ids,
    zeros of both signs, NaN among them. With cap 0.5 most of the larger values share a capped value."""
    rng = np.random.default_rng(V + k + B)
    low = np.finfo(np.float32).min
    x = (rng.standard_normal((B, V)) * 2).astype(np.float32)
    hists = []
    for b in range(B):
        r, few = x[b], rng.random(V) < 20.0 / V
        kind = b % 9
        if kind in (0, 1, 2):
            r[~few] = (-np.inf, -1e9, low)[kind]
        elif kind == 3:
            r[:] = rng.choice(np.array([0.0, -0.0, np.nan], np.float32), V)
        elif kind == 4:
            r[:] = (r > 1).astype(np.float32)
        elif kind == 5:
            r[:] = np.round(r)
        elif kind == 6:
            r[:] = np.round(r * 2) / 2
        elif kind == 7:                                    # many values and one, each in one part of the row
            r[: V // 2] = 3.0
        else:
            r[:] = np.where(rng.random(V) < 0.5, np.float32(7.0), np.nextafter(np.float32(7.0), np.float32(8.0)))
        hists.append(rng.integers(0, V, 0 if b % 3 else 400).astype(np.int32))
    p = mid_params(B, k, temperature=3.0, softcap=cap)
    p["repetition_penalty"][::3], p["frequency_penalty"][::3] = 1.3, 0.25
    p["top_p"][1::2] = 0.9
    check(x, p, hists, rng.random(B), kcap=2048)


def test_mid_k_more_penalised_ids_than_the_spill_list():
    rng = np.random.default_rng(5)
    V, H = 262144, 40000
    x = W.mixture_logits(rng, 2, V)
    p = mid_params(2, 100, frequency_penalty=0.3, repetition_penalty=1.1)
    p["temperature"][1] = 0.0
    check(x, p, [list(rng.permutation(V)[:H]) for _ in range(2)], rng.random(2), kcap=100)


@pytest.mark.parametrize("M,S,V", [(5, 8, 262144), (17, 3, 65537), (40, 2, 40000), (600, 1, 6000)])
def test_verify_windows_with_penalties(M, S, V):
    """Windows whose rows see their stream's history and the drafts fed before them, of equal and of ragged lengths."""
    rng = np.random.default_rng(M)
    for ragged in (False, True):
        m = np.full(S, M) if not ragged else np.maximum(1, M - np.arange(S) * 2 - 1)
        off = np.concatenate([[0], np.cumsum(m)]).astype(np.int64)
        R = int(off[-1])
        x = W.mixture_logits(rng, R, V)
        rows = x.argmax(axis=1).astype(np.int32)
        rows = np.where(rng.random(R) < 0.8, np.roll(rows, 1), rng.integers(0, V, R)).astype(np.int32)
        p = mid_params(S, 50, temperature=0.05, repetition_penalty=1.3)
        p["frequency_penalty"][::2] = 0.2
        p["repeat_last_n"][-1] = M // 2 + 1
        hist, hoff = csr([list(rng.integers(0, V, 5 + 7 * s)) for s in range(S)])
        u = rng.random(R)
        tok, acc = F.verify(torch.from_numpy(x).cuda(), rows, off, p, u=u, hist=hist, hist_off=hoff, eos_id=3)
        otok, oacc = O.verify(x, rows, off, hist, hoff, p, u, eos_id=3)
        np.testing.assert_array_equal(tok.cpu().numpy(), otok)
        np.testing.assert_array_equal(acc.cpu().numpy(), oacc)
        assert F.device_error() == 0


def test_mid_k_give_up_is_exact():
    """Segments that do not wait for each other: every sampled row is selected by its last segment alone, the tokens
    are the same and the give-up is reported; the next call finds clean counters."""
    from ferro_amd._lib import FS_DEVERR_INTERNAL, FS_WAIT_GIVE_UP
    rng = np.random.default_rng(9)
    B, V = 5, 65537
    x = W.mixture_logits(rng, B, V)
    p = mid_params(B, 300, repetition_penalty=1.2)
    p["frequency_penalty"][1] = 0.2
    p["temperature"][2] = 0.0
    hists = [list(W.zipf_ids(rng, V, 700)) for _ in range(B)]
    hist, off = csr(hists)
    u = rng.random(B)
    o = O.sample_batch(x, hist, off, p, u, kcap=300, nthreads=NT)
    ctx = F.sampler.Context()
    for limit, bits in ((FS_WAIT_GIVE_UP, FS_DEVERR_INTERNAL), (0, 0)):
        ctx.set_wait_limit(limit)
        out = F.sample_batch(torch.from_numpy(x).cuda(), p, u, hist=hist, hist_off=off, kcap=300, ctx=ctx)
        torch.cuda.synchronize()
        g = {k: v.cpu().numpy() for k, v in out.items() if v is not None and not k.startswith("_")}
        compare(g, o, p, u, 300)
        assert F.device_error(ctx) == bits


def test_mid_k_workspace_grows_by_need():
    """One context: batches that grow by a row and by what they need (penalties, every token a candidate, more segments), a
    small one after a large one."""
    rng = np.random.default_rng(11)
    ctx = F.sampler.Context()
    for B, V, k, rep in ((2, 70000, 100, 1.0), (3, 70000, 100, 1.2), (4, 70000, 0, 1.0), (5, 200000, 0, 1.3), (1, 33000, 300, 1.1),
                         (6, 33000, 70, 1.0), (7, 200000, 0, 1.2), (40, 33000, 90, 1.1), (3, 200000, 90, 1.1)):
        x = (rng.standard_normal((B, V)) * 2).astype(np.float32)
        p = mid_params(B, k, repetition_penalty=rep, frequency_penalty=0.01)
        hist, off = csr([rng.integers(0, V, 900).astype(np.int32) for _ in range(B)])
        u = rng.random(B)
        out = F.sample_batch(torch.from_numpy(x).cuda(), p, u, hist=hist, hist_off=off, ctx=ctx)
        torch.cuda.synchronize()
        o = O.sample_batch(x, hist, off, p, u, kcap=1, nthreads=NT)
        np.testing.assert_array_equal(out["tok"].cpu().numpy(), o["tok"])
        np.testing.assert_array_equal(out["keep"].cpu().numpy(), o["keep"])
        assert F.device_error(ctx) == 0


def test_mid_k_on_several_streams():
    """Three contexts on three streams, calls of few rows with the most segments each (they wait for each other) in
    flight together."""
    rng = np.random.default_rng(21)
    B, V = 9, 262144
    x = torch.from_numpy(W.mixture_logits(rng, B, V)).cuda()
    want, outs = [], []
    cfg = [(mid_params(B, k), rng.random(B), F.sampler.Context(), torch.cuda.Stream()) for k in (100, 0, 300)]
    cfg[1][0]["top_p"] = 0.9
    for p, u, ctx, _ in cfg:
        o = O.sample_batch(x.cpu().numpy(), np.zeros(0, np.int32), np.zeros(B + 1, np.int64), p, u, kcap=1, nthreads=NT)
        want.append(o["tok"])
        F.sample_batch(x, p, u, ctx=ctx)
    torch.cuda.synchronize()
    for _ in range(12):
        for i, (p, u, ctx, st) in enumerate(cfg):
            with torch.cuda.stream(st):
                outs.append((i, F.sample_batch(x, p, u, ctx=ctx)["tok"]))
    torch.cuda.synchronize()
    for i, tok in outs:
        np.testing.assert_array_equal(tok.cpu().numpy(), want[i])
    for _, _, ctx, _ in cfg:
        assert F.device_error(ctx) == 0


def test_mid_k_decode_steps():
    """Decode steps the mid-k kernel takes: history copies, draws and appends beside k > 64 and frequency penalties."""
    rng = np.random.default_rng(12)
    S, V = 6, 100004
    p = mid_params(S, 150, repetition_penalty=1.1, frequency_penalty=0.2)
    p["temperature"][1] = 0.0
    hist0 = [list(W.zipf_ids(rng, V, 300 * s)) for s in range(S)]
    rows = [W.mixture_logits(rng, S, V) for _ in range(4)]
    seeds = list(range(1, S + 1))
    want, want_hist, want_off = oracle_decode_loop(rows, p, seeds, hist0)
    d = F.DeviceRng(np.asarray(seeds, np.uint64))
    hist, off = (torch.from_numpy(a).cuda() for a in csr(hist0))
    for k, x in enumerate(rows):
        tok, _, hist, off = F.decode_step(torch.from_numpy(x).cuda(), p, d, hist=hist, hist_off=off)
        np.testing.assert_array_equal(tok.cpu().numpy(), want[k])
    np.testing.assert_array_equal(off.cpu().numpy(), want_off)
    np.testing.assert_array_equal(hist[:int(off[-1])].cpu().numpy(), want_hist)


@pytest.mark.parametrize("B,V", [(1, 4096), (3, 33001), (5, 65536), (24, 100003), (9, 262144), (70, 65537), (66, 262144)])
@pytest.mark.parametrize("top_p", [1.0, 0.95, 0.4])
def test_every_token_a_candidate(B, V, top_p):
    """top_k = 0 on every segment size: flat and spiky rows, bf16 values, narrow and wide spreads, all-equal and two-valued
    rows (no bin narrows them down), a masked vocabulary, infinities, NaN, a row without a number; penalties, a softcap,
    greedy and k <= 2048 rows among them."""
    rng = np.random.default_rng(V + B)
    x = (rng.standard_normal((B, V)) * 2).astype(np.float32)
    x[::2] = W.mixture_logits(rng, len(x[::2]), V)
    p = mid_params(B, 0, temperature=rng.uniform(0.5, 1.3, B))
    p["top_p"] = top_p
    p["repetition_penalty"][::3] = 1.2
    p["frequency_penalty"][1::4] = 0.2
    if B > 3:
        x[1] = bf16_valued(x[1])
        p["temperature"][2] = 0.0
        p["top_k"][3] = 80
    if B > 8:
        x[4, :] = 1.5                                # all equal
        x[5] = np.where(rng.random(V) < 0.5, 1.0, 2.0)
        x[6, rng.choice(V, V - 40, replace=False)] = -np.inf
        x[7] *= 1e-3
        x[8] = x[8] * 30 + 5
    if B > 20:
        x[9, 11] = np.inf
        x[10, :] = np.nan
        x[11, ::3] = np.nan
        x[12, :] = -np.inf
        x[13, 100] += 60.0                           # one token holds the whole mass
        p["softcap"][14:16] = 30.0
        x[15] *= 20
    u = rng.random(B)
    u[0] = 0.0
    hists = [list(W.zipf_ids(rng, V, int(rng.integers(0, 1500)))) for _ in range(B)]
    hist, off = csr(hists)
    out = F.sample_batch(torch.from_numpy(x).cuda(), p, u, hist=hist, hist_off=off)
    torch.cuda.synchronize()
    o = O.sample_batch(x, hist, off, p, u, kcap=1, nthreads=NT)
    np.testing.assert_array_equal(out["tok"].cpu().numpy(), o["tok"])
    np.testing.assert_array_equal(out["keep"].cpu().numpy(), o["keep"])
    assert F.device_error() == 0


@pytest.mark.parametrize("B,V", [(9, 4100), (9, 33000), (18, 100003), (9, 262144), (66, 262144)])
@pytest.mark.parametrize("cap", [0.0, 0.5])
def test_every_token_of_few_values(B, V, cap):
    """top_k = 0 on rows whose searched bins hold thousands of equal logits (located by value and count): one and two values,
    whole numbers, halves, zeros of both signs, two values in parts of the row, narrow rows below one large logit; with
    and without top-p, penalties on tied ids. With cap 0.5 most of the larger values share a capped value."""
    rng = np.random.default_rng(V + B)
    x = (rng.standard_normal((B, V)) * 2).astype(np.float32)
    hists = []
    for b in range(B):
        r, kind = x[b], b % 9
        if kind == 0:
            r[:] = 1.5
        elif kind == 1:
            r[:] = (r > 1).astype(np.float32)
        elif kind == 2:
            r[:] = np.round(r)
        elif kind == 3:
            r[:] = np.round(r * 2) / 2
        elif kind == 4:
            r[:] = rng.choice(np.array([0.0, -0.0, np.nan, -40.0], np.float32), V)
        elif kind == 5:
            r[: V // 2] = 3.0
        elif kind == 6:
            r[:] = np.maximum(r, 0)
        elif kind == 7:
            r[:] = r * 0.01
            r[V // 3] = 9.0
        else:
            r[rng.choice(V, V // 2, replace=False)] = -1e9
        hists.append(rng.integers(0, V, 0 if b % 2 else 300).astype(np.int32))
    p = mid_params(B, 0, temperature=0.9, softcap=cap)
    p["top_p"] = np.where(np.arange(B) % 4 < 2, 0.9, 1.0)
    p["repetition_penalty"][::2], p["frequency_penalty"][::4] = 1.3, 0.25
    u = rng.random(B)
    u[-1] = 0.0
    hist, off = csr(hists)
    out = F.sample_batch(torch.from_numpy(x).cuda(), p, u, hist=hist, hist_off=off)
    torch.cuda.synchronize()
    o = O.sample_batch(x, hist, off, p, u, kcap=1, nthreads=NT)
    np.testing.assert_array_equal(out["tok"].cpu().numpy(), o["tok"])
    np.testing.assert_array_equal(out["keep"].cpu().numpy(), o["keep"])
    assert F.device_error() == 0


@pytest.mark.parametrize("mask", [-np.inf, -1e9, np.finfo(np.float32).min])
def test_every_token_of_masked_rows_at_high_temperatures(mask):
    """Tokens masked far below rows that are narrow in units of the temperature: the bins cover the other tokens."""
    rng = np.random.default_rng(5)
    B, V = 10, 100003
    x = (rng.standard_normal((B, V)) * 2).astype(np.float32)
    x[::2, ::100] = mask
    x[1::2, :20000] = mask                           # whole segments of masked tokens
    x[4, 77777] = 6 * 3.0 * 32                       # the others are below the bins of this row
    x[5] = np.where(x[5] > 4, x[5], mask)
    x[2] = np.where(x[2] > 0, np.float32(2.0), mask)  # one value, the others masked: thousands, and a few
    x[3] = np.where(x[3] > 5.5, np.float32(2.0), mask)
    x[8:, 50001] = -130.0                            # one token below the bins of the others, one above its range
    x[9, 60000:] *= 0.01
    p = mid_params(B, 0, temperature=3.0)
    p["temperature"][6:8] = 0.7, 20.0
    p["top_p"] = np.where(np.arange(B) % 4 < 2, 0.9, 1.0)
    p["repetition_penalty"][::3] = 1.2
    hist, off = csr([rng.integers(0, V, 300).astype(np.int32) for _ in range(B)])
    for _ in range(3):
        u = rng.random(B)
        out = F.sample_batch(torch.from_numpy(x).cuda(), p, u, hist=hist, hist_off=off)
        torch.cuda.synchronize()
        o = O.sample_batch(x, hist, off, p, u, kcap=1, nthreads=NT)
        np.testing.assert_array_equal(out["tok"].cpu().numpy(), o["tok"])
        np.testing.assert_array_equal(out["keep"].cpu().numpy(), o["keep"])
    assert F.device_error() == 0


def test_every_token_draws_next_to_a_boundary():
    """Rows whose mass is ten logits, draws 6e-15 below and above the cumulative mass of each, computed in 80 bits. Ten
    masses summed in fp64 (or in units of 2^-52), each within 0.52 ulp, are off by less than 5e-15 of a sum >= 1; units of
    2^-44 would be off by up to 3e-14 each."""
    if np.finfo(np.longdouble).nmant < 63:
        pytest.skip("no 80-bit long double")
    rng = np.random.default_rng(44)
    B, V = 60, 40000
    x = np.full((B, V), -90.0, np.float32)
    p = mid_params(B, 0, temperature=1.0)
    p["top_p"] = 1.0
    u, want = np.zeros(B), np.zeros(B, np.int32)
    for b in range(B):
        at = rng.choice(V, 10, replace=False)
        x[b, at] = rng.uniform(-2, 0, 10).astype(np.float32)
        order = at[np.lexsort((at, -x[b, at]))]
        m = np.exp((x[b, order] - x[b].max()).astype(np.longdouble))
        c = np.cumsum(m)
        total = c[-1] + (V - 10) * np.exp(np.longdouble(-90.0) - np.longdouble(x[b].max()))
        j = int(rng.integers(2, 8))
        above = b % 2
        u[b] = float(c[j] / total * (1 + (6e-15 if above else -6e-15)))
        want[b] = order[j + above]
    out = F.sample_batch(torch.from_numpy(x).cuda(), p, u)
    np.testing.assert_array_equal(out["tok"].cpu().numpy(), want)


def test_every_token_give_up_and_decode():
    """Rows whose segments do not wait for each other are selected alone; decode steps and verification windows with
    top_k = 0."""
    from ferro_amd._lib import FS_DEVERR_INTERNAL, FS_WAIT_GIVE_UP
    rng = np.random.default_rng(3)
    S, V = 4, 40000
    p = mid_params(S, 0, temperature=0.8, repetition_penalty=1.1)
    p["top_p"][::2] = 0.9
    p["top_p"][1::2] = 1.0
    x = W.mixture_logits(rng, S, V)
    hists = [list(W.zipf_ids(rng, V, 400)) for _ in range(S)]
    hist, off = csr(hists)
    u = rng.random(S)
    o = O.sample_batch(x, hist, off, p, u, kcap=1, nthreads=NT)
    ctx = F.sampler.Context()
    for limit, bits in ((FS_WAIT_GIVE_UP, FS_DEVERR_INTERNAL), (0, 0)):
        ctx.set_wait_limit(limit)
        out = F.sample_batch(torch.from_numpy(x).cuda(), p, u, hist=hist, hist_off=off, ctx=ctx)
        torch.cuda.synchronize()
        np.testing.assert_array_equal(out["tok"].cpu().numpy(), o["tok"])
        np.testing.assert_array_equal(out["keep"].cpu().numpy(), o["keep"])
        assert F.device_error(ctx) == bits
    rows = [W.mixture_logits(rng, S, V) for _ in range(3)]
    seeds = list(range(1, S + 1))
    want, want_hist, want_off = oracle_decode_loop(rows, p, seeds, hists)
    d = F.DeviceRng(np.asarray(seeds, np.uint64))
    h, ho = torch.from_numpy(hist).cuda(), torch.from_numpy(off).cuda()
    for k, r in enumerate(rows):
        tok, _, h, ho = F.decode_step(torch.from_numpy(r).cuda(), p, d, hist=h, hist_off=ho)
        np.testing.assert_array_equal(tok.cpu().numpy(), want[k])
    np.testing.assert_array_equal(h[:int(ho[-1])].cpu().numpy(), want_hist)
    R = 12
    xv = W.mixture_logits(rng, R, V)
    fed = xv.argmax(axis=1).astype(np.int32)
    ro = np.array([0, 3, 4, 9, 12], np.int64)
    uv = rng.random(R)
    tok, acc = F.verify(torch.from_numpy(xv).cuda(), fed, ro, p, u=uv, hist=hist, hist_off=off)
    otok, oacc = O.verify(xv, fed, ro, hist, off, p, uv)
    np.testing.assert_array_equal(tok.cpu().numpy(), otok)
    np.testing.assert_array_equal(acc.cpu().numpy(), oacc)


@pytest.mark.parametrize("every", [False, True])
@pytest.mark.parametrize("warm", [True, False])
def test_mid_k_calls_in_a_graph(every, warm):
    """fs_sample_batch_hp recorded into a graph and replayed, with eager calls of another size between the replays: the
    counters, lists and mass bins are left as each replay needs them. A context that never ran such a batch takes the
    fused kernel under capture (no allocation there): the same tokens."""
    import ctypes
    from ferro_amd._lib import lib
    from test_gpu_graph import Call, P, check_clean, mixed
    B, V = 40, 65536
    ctx, other = F.sampler.Context(), F.sampler.Context()
    ws = [mixed(31 + i, B, V) for i in range(3)]
    for w in ws:
        w.params["top_k"][w.params["top_k"] == 0] = 0 if every else 1500
    calls = [Call(w, kcap=16) for w in ws]

    def launch(i, c, st):
        outs = (None, None) if every else (P(calls[i].ids), P(calls[i].probs))
        rc = lib().fs_sample_batch_hp(c.h, P(calls[i].x), calls[i].x.stride(0), B if i < 2 else B // 2, V, P(calls[i].hist),
                                      P(calls[i].hoff), P(calls[i].params),
                                      ws[i].params.ctypes.data_as(ctypes.c_void_p), P(calls[i].u), P(calls[i].tok),
                                      0 if every else 16, *outs, P(calls[i].keep), ctypes.c_void_p(st.cuda_stream))
        assert rc == 0, rc

    cur, side = torch.cuda.current_stream(), torch.cuda.Stream()
    want = []
    for i in range(2):
        calls[i].poison()
        launch(i, ctx if warm else other, cur)
        torch.cuda.synchronize()
        want.append(calls[i].out())
    if not warm:                                       # (the fused kernel's workspace only)
        F.sample_batch(calls[0].x[:, :V], ws[0].params, ws[0].u, hist=ws[0].hist, hist_off=ws[0].hist_off, ctx=ctx,
                       route="device")
        torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    side.wait_stream(cur)
    with torch.cuda.stream(side):
        with torch.cuda.graph(g, stream=side):
            for i in range(2):
                launch(i, ctx, side)
    cur.wait_stream(side)
    torch.cuda.synchronize()
    for rep in range(3):
        for c in calls[:2]:
            c.poison()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        for i in range(2):
            got = calls[i].out()
            for k in ("tok", "keep", "ids"):
                np.testing.assert_array_equal(got[k], want[i][k], err_msg=f"replay {rep} call {i} {k}")
            np.testing.assert_allclose(got["probs"], want[i]["probs"], rtol=1e-12)   # (sums in another order)
        launch(2, ctx, cur)
        torch.cuda.synchronize()
        check_clean(ctx)
    del g


@pytest.mark.parametrize("params", [dict(min_p=0.05, top_k=0), dict(top_k=3000)])
def test_recorded_call_the_mid_k_kernel_refuses(params):
    """A context warmed up with a batch of the mid-k kernel records the same shape with parameters that only the fused
    kernel takes: its workspace is there, nothing is allocated in the capture."""
    import ctypes
    from ferro_amd._lib import lib
    from test_gpu_graph import Call, P, check_clean, mixed
    B, V = 24, 65536
    ctx, other = F.sampler.Context(), F.sampler.Context()
    warm, w = mixed(3, B, V), mixed(4, B, V)
    warm.params["top_k"][:], warm.params["min_p"][:] = 0, 0.0
    for f, v in params.items():
        w.params[f][:] = v

    def launch(c, wl, call, st):
        rc = lib().fs_sample_batch_hp(c.h, P(call.x), call.x.stride(0), B, V, P(call.hist), P(call.hoff), P(call.params),
                                      wl.params.ctypes.data_as(ctypes.c_void_p), P(call.u), P(call.tok), 0, None, None,
                                      P(call.keep), ctypes.c_void_p(st.cuda_stream))
        assert rc == 0, rc

    cw, c = Call(warm, kcap=16), Call(w, kcap=16)
    cur, side = torch.cuda.current_stream(), torch.cuda.Stream()
    launch(ctx, warm, cw, cur)
    launch(other, w, c, cur)
    torch.cuda.synchronize()
    want = c.out()
    g = torch.cuda.CUDAGraph()
    side.wait_stream(cur)
    with torch.cuda.stream(side):
        with torch.cuda.graph(g, stream=side):
            launch(ctx, w, c, side)
    cur.wait_stream(side)
    torch.cuda.synchronize()
    for rep in range(3):
        c.poison()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        got = c.out()
        for k in ("tok", "keep"):
            np.testing.assert_array_equal(got[k], want[k], err_msg=f"replay {rep} {k}")
        launch(ctx, warm, cw, cur)
        torch.cuda.synchronize()
        check_clean(ctx)
    del g
