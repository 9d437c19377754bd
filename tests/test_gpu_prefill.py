"""GPU parity: ragged paged prefill attention (MFMA) vs the fp32 oracle.

Tolerance (the ``parity`` fixture): max-abs 2e-2 against the fp32 oracle on
bf16 inputs, and max |out - ref| / max(1, |ref|) <= 1.2e-2; each case's errors
are printed in the session's parity table.
"""

from __future__ import annotations

import pytest
import torch

from oracle import attention as oatt
from tests.helpers import make_paged_batch

pytestmark = pytest.mark.gpu


def _run(dev, b, qo_lens, hq, hkv, d, causal=True, seed=0):
    from minimal_inference_amd.prefill import BatchPrefillWithPagedKVCacheWrapper

    g = torch.Generator().manual_seed(seed)
    total = sum(qo_lens)
    q = torch.randn(total, hq, d, generator=g).to(torch.bfloat16)
    qo = [0]
    for x in qo_lens:
        qo.append(qo[-1] + x)
    ws = torch.empty(64 << 20, dtype=torch.uint8, device=dev)
    w = BatchPrefillWithPagedKVCacheWrapper(ws, "NHD")
    qo_d = torch.tensor(qo, dtype=torch.int32, device=dev)
    ip = torch.tensor(b["indptr"], dtype=torch.int32, device=dev)
    lp = torch.tensor(b["last"], dtype=torch.int32, device=dev)
    ix = b["indices"].to(dev)
    w.plan(qo_d, ip, ix, lp, hq, hkv, d, 16, causal=causal, pos_encoding_mode="NONE",
           q_data_type=torch.bfloat16)
    out = w.run(q.to(dev), b["pool"].to(dev))
    torch.cuda.synchronize()
    ref = oatt.prefill(q, b["pool"], qo, b["indptr"], b["indices"].tolist(), b["last"], causal=causal)
    return out.float().cpu(), ref


@pytest.mark.parametrize("hq,hkv,d", [(14, 2, 64), (32, 8, 128), (28, 4, 128), (64, 8, 128),
                                      (6, 3, 128), (8, 1, 64), (16, 4, 256), (8, 1, 256), (10, 2, 256),
                                      (40, 8, 128)])
@pytest.mark.parametrize("L", [1, 5, 64, 100, 300])
def test_single_request_causal(dev, parity, hq, hkv, d, L):
    b = make_paged_batch([L], hq, hkv, d, seed=L + d)
    out, ref = _run(dev, b, [L], hq, hkv, d, seed=L)
    parity(out, ref)


def test_ragged_batch(dev, parity):
    lens = [37, 200, 5, 513, 64, 1]
    b = make_paged_batch(lens, 32, 8, 128, seed=9)
    out, ref = _run(dev, b, lens, 32, 8, 128, seed=9)
    parity(out, ref)


@pytest.mark.parametrize("hq,hkv,d", [(28, 4, 128), (14, 2, 64), (64, 8, 128), (16, 4, 256)])
def test_kv_longer_than_q_bottom_right_causal(dev, parity, hq, hkv, d):
    """Chunked-prefill shape: the last qo_len of kv_len tokens are queries
    (row blocks whose diagonal starts mid-tile, at every head_dim and group 8)."""
    kv_lens = [100, 260, 33]
    qo_lens = [20, 64, 33]
    b = make_paged_batch(kv_lens, hq, hkv, d, seed=4)
    out, ref = _run(dev, b, qo_lens, hq, hkv, d, seed=4)
    parity(out, ref)


@pytest.mark.parametrize("hq,hkv,d", [(32, 8, 128), (14, 2, 64)])
def test_zero_length_query_spans_in_a_ragged_batch(dev, parity, hq, hkv, d):
    """Requests with no query rows -- one with cached tokens, one empty --
    between requests with rows (one of them chunked: 10 rows over 64 tokens)
    get no tiles, and the rows around them are unaffected."""
    kv_lens = [37, 200, 0, 64, 1]
    qo_lens = [37, 0, 0, 10, 1]
    b = make_paged_batch(kv_lens, hq, hkv, d, seed=41)
    out, ref = _run(dev, b, qo_lens, hq, hkv, d, seed=41)
    assert out.shape[0] == sum(qo_lens)
    parity(out, ref)


@pytest.mark.parametrize("sm_scale", [0.3, 0.02])
def test_explicit_softmax_scale(dev, parity, sm_scale):
    """plan(sm_scale=...) replaces 1/sqrt(head_dim) in the causal prefill."""
    from minimal_inference_amd.prefill import BatchPrefillWithPagedKVCacheWrapper

    hq, hkv, d = 32, 8, 128
    lens = [37, 300, 5]
    b = make_paged_batch(lens, hq, hkv, d, seed=58)
    g = torch.Generator().manual_seed(58)
    q = torch.randn(sum(lens), hq, d, generator=g).to(torch.bfloat16)
    qo = [0]
    for x in lens:
        qo.append(qo[-1] + x)
    w = BatchPrefillWithPagedKVCacheWrapper(torch.empty(64 << 20, dtype=torch.uint8, device=dev), "NHD")
    w.plan(torch.tensor(qo, dtype=torch.int32, device=dev), torch.tensor(b["indptr"], dtype=torch.int32, device=dev),
           b["indices"].to(dev), torch.tensor(b["last"], dtype=torch.int32, device=dev), hq, hkv, d, 16,
           causal=True, sm_scale=sm_scale)
    out = w.run(q.to(dev), b["pool"].to(dev)).float().cpu()
    ref = oatt.prefill(q, b["pool"], qo, b["indptr"], b["indices"].tolist(), b["last"], causal=True,
                       sm_scale=sm_scale)
    parity(out, ref)


@pytest.mark.parametrize("hq,hkv,d", [(32, 8, 128), (14, 2, 64)])
def test_large_scores_lazy_rescale(dev, parity, hq, hkv, d):
    """q and K scaled by 6: the row maxima grow past the lazy
    rescale margin many times along a row's key tiles."""
    lens = [300, 777]
    b = make_paged_batch(lens, hq, hkv, d, seed=62)
    b["pool"][:, 0] = (b["pool"][:, 0].float() * 6).to(torch.bfloat16)
    # V / 4 keeps the near one-hot outputs (single V entries) near unit size,
    # where the max-abs bound applies
    b["pool"][:, 1] = (b["pool"][:, 1].float() / 4).to(torch.bfloat16)
    from minimal_inference_amd.prefill import BatchPrefillWithPagedKVCacheWrapper

    g = torch.Generator().manual_seed(62)
    q = (torch.randn(sum(lens), hq, d, generator=g) * 6).to(torch.bfloat16)
    qo = [0]
    for x in lens:
        qo.append(qo[-1] + x)
    w = BatchPrefillWithPagedKVCacheWrapper(torch.empty(64 << 20, dtype=torch.uint8, device=dev), "NHD")
    w.plan(torch.tensor(qo, dtype=torch.int32, device=dev), torch.tensor(b["indptr"], dtype=torch.int32, device=dev),
           b["indices"].to(dev), torch.tensor(b["last"], dtype=torch.int32, device=dev), hq, hkv, d, 16, causal=True)
    out = w.run(q.to(dev), b["pool"].to(dev)).float().cpu()
    assert torch.isfinite(out).all()
    ref = oatt.prefill(q, b["pool"], qo, b["indptr"], b["indices"].tolist(), b["last"], causal=True)
    parity(out, ref)


@pytest.mark.parametrize("hq,hkv,d", [(32, 8, 128), (14, 2, 64), (16, 4, 256)])
def test_head_major_q_and_out_views(dev, parity, hq, hkv, d):
    """q and out as head-major views ([heads, rows, head_dim] storage seen as
    [rows, heads, head_dim]: a head stride of rows * head_dim, larger than
    the row stride), as a single prompt's q.permute(0, 2, 1, 3).reshape(...)
    is when q is a contiguous [1, heads, seq, head_dim] tensor; every tile's
    rows and heads are read and written through them."""
    from minimal_inference_amd.prefill import BatchPrefillWithPagedKVCacheWrapper

    lens = [37, 300, 5, 129]
    b = make_paged_batch(lens, hq, hkv, d, seed=47)
    g = torch.Generator().manual_seed(47)
    q = torch.randn(sum(lens), hq, d, generator=g).to(torch.bfloat16)
    qo = [0]
    for x in lens:
        qo.append(qo[-1] + x)
    w = BatchPrefillWithPagedKVCacheWrapper(torch.empty(64 << 20, dtype=torch.uint8, device=dev), "NHD")
    w.plan(torch.tensor(qo, dtype=torch.int32, device=dev), torch.tensor(b["indptr"], dtype=torch.int32, device=dev),
           b["indices"].to(dev), torch.tensor(b["last"], dtype=torch.int32, device=dev), hq, hkv, d, 16, causal=True)
    q_hm = q.transpose(0, 1).contiguous().to(dev).transpose(0, 1)
    out_hm = torch.full((hq, sum(lens), d), float("nan"), dtype=torch.bfloat16, device=dev).transpose(0, 1)
    assert q_hm.stride() == (d, sum(lens) * d, 1) and out_hm.stride() == q_hm.stride()
    got = w.run(q_hm, b["pool"].to(dev), out=out_hm)
    assert got.data_ptr() == out_hm.data_ptr()
    ref = oatt.prefill(q, b["pool"], qo, b["indptr"], b["indices"].tolist(), b["last"], causal=True)
    out = out_hm.float().cpu()
    assert torch.isfinite(out).all()
    parity(out, ref)


@pytest.mark.parametrize("hq,hkv,d", [(16, 4, 64), (32, 8, 128), (28, 4, 128), (16, 4, 256)])
def test_non_causal(dev, parity, hq, hkv, d):
    lens = [50, 129, 1, 300]
    b = make_paged_batch(lens, hq, hkv, d, seed=6)
    out, ref = _run(dev, b, lens, hq, hkv, d, causal=False, seed=6)
    parity(out, ref)


@pytest.mark.parametrize("hq,hkv,d", [(32, 8, 128), (14, 2, 64)])
def test_non_causal_kv_longer_than_q(dev, parity, hq, hkv, d):
    """Non-causal rows over a longer cached context: every row sees every
    key, including the keys past its own position."""
    kv_lens = [100, 260, 33]
    qo_lens = [20, 64, 1]
    b = make_paged_batch(kv_lens, hq, hkv, d, seed=44)
    out, ref = _run(dev, b, qo_lens, hq, hkv, d, causal=False, seed=44)
    parity(out, ref)


def test_first_row_attends_only_to_token0(dev):
    """Causal row 0 sees one key, so its output is V[0] of its KV head."""
    b = make_paged_batch([40], 8, 2, 128, seed=12)
    out, _ = _run(dev, b, [40], 8, 2, 128, seed=12)
    page0 = int(b["indices"][0])
    v0 = b["pool"][page0, 1, 0].float().repeat_interleave(4, dim=0)
    assert torch.equal(out[0], v0)


def test_prefill_then_decode_consistency(dev, parity):
    """The last prefill row equals a decode query over the same context."""
    from minimal_inference_amd.decode import BatchDecodeWithPagedKVCacheWrapper

    lens = [77, 130]
    b = make_paged_batch(lens, 32, 8, 128, seed=15)
    out, _ = _run(dev, b, lens, 32, 8, 128, seed=15)
    g = torch.Generator().manual_seed(15)
    q = torch.randn(sum(lens), 32, 128, generator=g).to(torch.bfloat16)
    last_q = torch.stack([q[76], q[77 + 129]])
    ws = torch.empty(64 << 20, dtype=torch.uint8, device=dev)
    w = BatchDecodeWithPagedKVCacheWrapper(ws)
    w.plan(torch.tensor(b["indptr"], dtype=torch.int32, device=dev), b["indices"].to(dev),
           torch.tensor(b["last"], dtype=torch.int32, device=dev), 32, 8, 128, 16)
    dec = w.run(last_q.to(dev), b["pool"].to(dev)).float().cpu()
    parity(dec, torch.stack([out[76], out[77 + 129]]))


def _poison_tails(b):
    """NaN in every row past each request's length on its last page (K and V),
    where a pool holds stale data in practice; no result may read them."""
    pool = b["pool"].clone()
    idx = b["indices"].tolist()
    for r in range(len(b["last"])):
        lo, hi = b["indptr"][r], b["indptr"][r + 1]
        if hi > lo and b["last"][r] < 16:
            pool[idx[hi - 1], :, b["last"][r]:] = float("nan")
    return {**b, "pool": pool}


@pytest.mark.parametrize("hq,hkv,d", [(32, 8, 128), (14, 2, 64)])
def test_stale_rows_past_the_end_are_not_read(dev, parity, hq, hkv, d):
    lens = [37, 100, 5, 250]
    b = _poison_tails(make_paged_batch(lens, hq, hkv, d, seed=21))
    out, ref = _run(dev, b, lens, hq, hkv, d, seed=21)
    assert torch.isfinite(out).all()
    parity(out, ref)


def test_long_prompt_4096(dev, parity):
    """One 4,096-token causal prompt: 64 key tiles for the last query rows,
    the longest per-workgroup loop the bench batches do not reach."""
    b = make_paged_batch([4096], 8, 2, 128, seed=41)
    out, ref = _run(dev, b, [4096], 8, 2, 128, seed=41)
    parity(out, ref)


# (heads, new rows per request, cached tokens per request, row blocks per wave the plan picks)
SPLIT_CASES = [
    ((32, 8, 128), [3], [1000], 1),             # one short tile per KV head, cut at kMinChunk
    ((28, 4, 128), [193, 1, 64], [900, 65, 0], 1),  # fine tiles, ragged, one that is not split
    ((8, 1, 64), [2], [9000], 1),               # a single tile: the most units one merge takes
    ((64, 8, 128), [200, 37], [5001, 3000], 3),  # coarse tiles of three row blocks
    ((14, 2, 64), [700], [4010], 2),
    ((16, 4, 256), [70], [2500], 1),
]


@pytest.mark.parametrize("heads,qo_lens,cached,blocks", SPLIT_CASES)
@pytest.mark.parametrize("causal", [True, False])
def test_tiles_split_over_the_keys(dev, parity, heads, qo_lens, cached, blocks, causal):
    """Tiles cut into units along the keys: against the oracle, the same bits
    on every run of a plan (the merge counters are back at zero), and with a
    workspace that has no room for partials (nothing is split)."""
    from minimal_inference_amd import _lib
    from minimal_inference_amd.prefill import BatchPrefillWithPagedKVCacheWrapper

    hq, hkv, d = heads
    b = make_paged_batch([q + c for q, c in zip(qo_lens, cached)], hq, hkv, d, seed=17)
    total = sum(qo_lens)
    q = torch.randn(total, hq, d, generator=torch.Generator().manual_seed(17)).to(torch.bfloat16)
    qo = [0]
    for n in qo_lens:
        qo.append(qo[-1] + n)
    args = [torch.tensor(qo, dtype=torch.int32, device=dev), torch.tensor(b["indptr"], dtype=torch.int32, device=dev),
            b["indices"].to(dev), torch.tensor(b["last"], dtype=torch.int32, device=dev)]
    qd, pool = q.to(dev), b["pool"].to(dev)
    ref = oatt.prefill(q, b["pool"], qo, b["indptr"], b["indices"].tolist(), b["last"], causal=causal)

    def run(nbytes):
        ws = torch.full((nbytes,), 0x5a, dtype=torch.uint8, device=dev)
        w = BatchPrefillWithPagedKVCacheWrapper(ws, "NHD")
        w.plan(*args, hq, hkv, d, 16, causal=causal, max_total_q=total)
        outs = [w.run(qd, pool).cpu() for _ in range(3)]
        return ws[:32].view(torch.int32).tolist(), outs

    header, outs = run(128 << 20)
    assert header[1] == 0 and header[3] == blocks and header[4] > 0  # no error, the form, a split
    parity(outs[0].float(), ref)
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
    header, whole = run(int(_lib.load().mi_prefill_workspace_size(len(qo_lens), total)))
    assert header[1] == 0 and header[4] == 0
    parity(whole[0].float(), ref)


class _Planned:
    """A batch on the GPU, and what runs of its plan give that take whole tiles
    (a workspace of the least size) and that take the units."""

    def __init__(self, dev, heads, qo_lens, cached, seed):
        from minimal_inference_amd import _lib

        self.dev, self.heads, self.total = dev, heads, sum(qo_lens)
        hq, hkv, d = heads
        b = make_paged_batch([q + c for q, c in zip(qo_lens, cached)], hq, hkv, d, seed=seed)
        qo = [0]
        for n in qo_lens:
            qo.append(qo[-1] + n)
        self.batch = len(qo_lens)
        self.csr = [torch.tensor(qo, dtype=torch.int32, device=dev), torch.tensor(b["indptr"], dtype=torch.int32, device=dev),
                    b["indices"].to(dev), torch.tensor(b["last"], dtype=torch.int32, device=dev)]
        self.pool = b["pool"].to(dev)
        g = torch.Generator(device=dev).manual_seed(seed)
        self.q = [torch.randn(self.total, hq, d, device=dev, generator=g).to(torch.bfloat16) for _ in range(3)]
        self.need = int(_lib.load().mi_prefill_workspace_size(self.batch, self.total))
        self.w, self.ws = self.plan(128 << 20)
        self.units = [self.w.run(q, self.pool) for q in self.q]
        small, _ = self.plan(self.need)
        self.whole = [small.run(q, self.pool) for q in self.q]
        torch.cuda.synchronize()

    def plan(self, nbytes, ws=None):
        from minimal_inference_amd.prefill import BatchPrefillWithPagedKVCacheWrapper

        ws = torch.full((nbytes,), 0x5a, dtype=torch.uint8, device=self.dev) if ws is None else ws
        w = BatchPrefillWithPagedKVCacheWrapper(ws, "NHD")
        w.plan(*self.csr, *self.heads, 16, causal=True, max_total_q=self.total)
        return w, ws

    def run_abi(self, ws, q, pool, heads):
        """mi_prefill_run of whatever plan `ws` holds."""
        from minimal_inference_amd import _lib

        out = torch.empty_like(q)
        _lib.call("mi_prefill_run", ws.data_ptr(), ws.numel(), q.data_ptr(), q.stride(0), q.stride(1), pool.data_ptr(),
                  pool.shape[0], self.csr[2].data_ptr(), out.data_ptr(), out.stride(0), out.stride(1), self.batch,
                  self.total, *heads, 16, 1, 0.0, torch.cuda.current_stream().cuda_stream)
        return out


OWNED_CASES = [((32, 8, 128), [3], [1000]), ((64, 8, 128), [200, 37], [5001, 3000]), ((14, 2, 64), [700], [4010]),
               ((16, 4, 256), [70], [2500])]


@pytest.mark.parametrize("heads,qo_lens,cached", OWNED_CASES)
def test_runs_outside_of_the_plans_stream_only_read_the_workspace(dev, heads, qo_lens, cached):
    """Runs of one plan that nothing orders: those on other streams than the
    plan's and those of a graph take whole tiles and leave every byte of the
    workspace alone, so they may overlap each other and one on the plan's
    stream."""
    c = _Planned(dev, heads, qo_lens, cached, seed=31)
    assert not torch.equal(c.units[0], c.whole[0])  # (split rows round differently)
    before = c.ws.clone()
    torch.cuda.synchronize()
    sides = [torch.cuda.Stream(), torch.cuda.Stream()]
    for s in sides:
        with torch.cuda.stream(s):
            out = c.w.run(c.q[0], c.pool)
        s.synchronize()
        assert torch.equal(out, c.whole[0])
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = c.w.run(c.q[1], c.pool)
    for _ in range(3):
        captured.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(captured, c.whole[1]) and torch.equal(c.ws, before)
        assert torch.equal(c.w.run(c.q[1], c.pool), c.units[1])
        before = c.ws.clone()
    # all of them at once
    outs = []
    for i in range(12):
        outs.append((c.w.run(c.q[i % 3], c.pool), c.units[i % 3]))
        for k, s in enumerate(sides):
            with torch.cuda.stream(s):
                outs.append((c.w.run(c.q[(i + k) % 3], c.pool), c.whole[(i + k) % 3]))
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in outs)


@pytest.mark.parametrize("heads,qo_lens,cached", OWNED_CASES)
def test_saved_plans_and_other_geometry_take_whole_tiles(dev, heads, qo_lens, cached):
    """A plan's bytes in another buffer (whole, or the documented least size), put
    back over a later plan's, or run with other head counts of the same group:
    the partials belong to the plan in place, so these runs take whole tiles and
    write nothing but the output."""
    c = _Planned(dev, heads, qo_lens, cached, seed=32)
    saved = c.ws[:c.need].clone()
    for copy in (c.ws.clone(), saved.clone()):
        kept = copy.clone()
        assert torch.equal(c.run_abi(copy, c.q[0], c.pool, heads), c.whole[0])
        assert torch.equal(copy, kept)
    assert torch.equal(c.run_abi(c.ws, c.q[0], c.pool, heads), c.units[0])  # (in place)
    other = _Planned(dev, heads, [n + 5 for n in qo_lens], cached, seed=33)
    other.plan(0, ws=c.ws)
    c.ws[:c.need].copy_(saved)
    kept = c.ws.clone()
    assert torch.equal(c.run_abi(c.ws, c.q[0], c.pool, heads), c.whole[0])
    assert torch.equal(c.ws, kept)
    # twice the heads, in groups of the same size
    hq, hkv, d = heads
    q2, pool2 = torch.cat([c.q[0], c.q[1]], 1), torch.cat([c.pool, c.pool.flip(0)], 3)
    c.plan(0, ws=c.ws)
    kept = c.ws.clone()
    out2 = c.run_abi(c.ws, q2, pool2, (2 * hq, 2 * hkv, d))
    assert torch.equal(out2[:, :hq], c.whole[0])
    flipped, _ = c.plan(c.need)
    assert torch.equal(out2[:, hq:], flipped.run(c.q[1], pool2[:, :, :, hkv:].contiguous()))
    assert torch.equal(c.ws, kept)
