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


# (heads, new rows per request, cached tokens per request, row blocks per wave the
# plan picks, KV tiles per unit at most, units)
SPLIT_CASES = [
    ((32, 8, 128), [3], [1000], 1, 4, 4),             # one short tile per KV head, cut at kMinChunk
    ((28, 4, 128), [193, 1, 64], [900, 65, 0], 1, 4, 106),  # fine tiles, ragged, some that are not split
    ((8, 1, 64), [2], [9000], 1, 8, 18),              # a single tile of 141 KV tiles, cut at sqrt(141 / 2)
    ((64, 8, 128), [200, 37], [5001, 3000], 3, 14, 62),  # coarse tiles of three row blocks
    ((14, 2, 64), [700], [4010], 2, 8, 353),
    ((16, 4, 256), [70], [2500], 1, 4, 52),
    # more tiles than the plan's block has threads, over two resident rounds, the last one split
    ((8, 1, 64), [144] * 60 + [8], [0] * 60 + [9000], 1, 8, 1098),
]


@pytest.mark.parametrize("heads,qo_lens,cached,blocks,chunk,units", SPLIT_CASES)
@pytest.mark.parametrize("causal", [True, False])
def test_tiles_split_over_the_keys(dev, parity, heads, qo_lens, cached, blocks, chunk, units, causal):
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
    assert header[1] == 0 and header[3] == blocks and header[4] == chunk and header[6] == units
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


def test_few_partial_slots_bind_the_split(dev, parity):
    """A workspace with room for two slots of coarse units (five of fine ones): two
    tiles of 32 KV tiles that are cut into eight units each where there is room are
    cut into two, and merged from them."""
    c = _Planned(dev, (32, 8, 128), [20], [2000], seed=34)
    assert c.ws[16:28].view(torch.int32).tolist()[::2] == [4, 16]  # chunk, units
    w, ws = c.plan(2300 << 10)
    assert ws[16:28].view(torch.int32).tolist()[::2] == [16, 4]
    outs = [w.run(c.q[0], c.pool) for _ in range(3)]
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
    assert not torch.equal(outs[0], c.whole[0])
    parity(outs[0].float().cpu(), c.whole[0].float().cpu())


def test_more_requests_than_the_plans_threads(dev, parity):
    """1,100 requests of 1 to 40 rows, some of none, some on cached tokens."""
    g = torch.Generator().manual_seed(35)
    qo_lens = torch.randint(0, 41, (1100,), generator=g).tolist()
    kv_lens = [n + (100 if i % 7 == 0 else 0) for i, n in enumerate(qo_lens)]
    b = make_paged_batch(kv_lens, 4, 2, 64, seed=35)
    out, ref = _run(dev, b, qo_lens, 4, 2, 64, seed=35)
    parity(out, ref)


@pytest.mark.parametrize("batch", [1100, 300])
def test_a_list_too_short_for_the_rows_counts_whole_requests(dev, batch):
    """A plan told of fewer rows than qo_indptr has reports the error, and counts
    only tiles that it has written: those of the requests that fit."""
    from minimal_inference_amd.prefill import BatchPrefillWithPagedKVCacheWrapper

    qo = torch.arange(batch + 1, dtype=torch.int32, device=dev) * 40  # three tiles of 16 rows each
    pages = torch.arange(batch + 1, dtype=torch.int32, device=dev) * 3
    ws = torch.full((1 << 20,), 0x5a, dtype=torch.uint8, device=dev)
    w = BatchPrefillWithPagedKVCacheWrapper(ws, "NHD")
    w.plan(qo, pages, torch.zeros(3 * batch, dtype=torch.int32, device=dev),
           torch.full((batch,), 8, dtype=torch.int32, device=dev), 8, 1, 64, 16, causal=True, max_total_q=104)
    capacity = 104 // 8 + batch + 1
    num_tiles, error = ws[:8].view(torch.int32).tolist()
    assert error == 1 and num_tiles == capacity // 3 * 3 and capacity % 3
    records = ws[256:256 + 32 * (num_tiles + 1)].view(torch.int32).view(-1, 8).cpu()
    assert bool((records[:num_tiles, 2] == 40).all()) and int(records[num_tiles, 2]) != 40


@pytest.mark.parametrize("heads,qo_lens,cached", OWNED_CASES)
def test_split_tiles_with_head_major_rows(dev, heads, qo_lens, cached):
    """q and out with other strides on split tiles of every form: head-major, and
    rows further apart than their heads; the bits of contiguous ones, nothing
    written between the rows."""
    c = _Planned(dev, heads, qo_lens, cached, seed=36)
    hq, _, d = heads
    q = c.q[0].transpose(0, 1).contiguous().transpose(0, 1)
    out = torch.full((hq, c.total, d), float("nan"), dtype=torch.bfloat16, device=dev).transpose(0, 1)
    c.w.run(q, c.pool, out=out)
    assert torch.equal(out, c.units[0])
    wide = torch.full((c.total, hq + 3, d + 8), 7.0, dtype=torch.bfloat16, device=dev)
    wide_q = wide.clone()
    wide_q[:, 1:1 + hq, :d] = c.q[0]
    c.w.run(wide_q[:, 1:1 + hq, :d], c.pool, out=wide[:, 2:2 + hq, :d])
    assert torch.equal(wide[:, 2:2 + hq, :d], c.units[0])
    wide[:, 2:2 + hq, :d] = 7.0
    assert bool((wide == 7.0).all())


def test_plans_with_and_without_units_under_one_graph(dev):
    """Plans in turn that split and do not, in one workspace, each followed by an
    eager run and a replay of the run captured under the first."""
    split = _Planned(dev, (32, 8, 128), [40, 3], [2000, 1000], seed=37)
    flat = _Planned(dev, (32, 8, 128), [20, 23], [0, 30], seed=38)
    split.plan(0, ws=split.ws)
    q, pool = split.q[0].clone(), torch.zeros(max(split.pool.shape[0], flat.pool.shape[0]), *split.pool.shape[1:],
                                              dtype=torch.bfloat16, device=dev)
    indices = torch.zeros(max(split.csr[2].numel(), flat.csr[2].numel()), dtype=torch.int32, device=dev)
    static = [t.clone() for t in split.csr[:2]] + [indices, split.csr[3].clone()]
    w = split.w
    w.plan(*static, 32, 8, 128, 16, causal=True, max_total_q=split.total)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = w.run(q, pool)
    for c in (split, flat, split, split, flat, flat, split):
        for t, v in zip(static, c.csr):
            t[:v.numel()].copy_(v)
        pool[:c.pool.shape[0]].copy_(c.pool)
        w.plan(*static, 32, 8, 128, 16, causal=True, max_total_q=c.total)
        assert (int(w._ws[16:20].view(torch.int32)[0]) > 0) == (c is split)
        for k in range(2):
            q.copy_(c.q[k])
            graph.replay()
            assert torch.equal(captured, c.whole[k])
            assert torch.equal(w.run(q, pool), c.units[k])


def test_plan_and_run_captured_together(dev):
    """A captured plan lists whole tiles only, on every replay and for the eager runs
    after it, whatever an eager plan left in the workspace."""
    split = _Planned(dev, (32, 8, 128), [40, 3], [2000, 1000], seed=37)
    static, q = [t.clone() for t in split.csr], split.q[0].clone()
    w = split.w
    w.plan(*static, 32, 8, 128, 16, causal=True, max_total_q=split.total)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        w.plan(*static, 32, 8, 128, 16, causal=True, max_total_q=split.total)
        captured = w.run(q, split.pool)
    for k in range(3):
        q.copy_(split.q[k])
        graph.replay()
        assert torch.equal(captured, split.whole[k])
        assert torch.equal(w.run(q, split.pool), split.whole[k])
        w.plan(*static, 32, 8, 128, 16, causal=True, max_total_q=split.total)
        assert torch.equal(w.run(q, split.pool), split.units[k])


@pytest.mark.parametrize("heads,qo_lens,cached", OWNED_CASES)
def test_infinities_and_nan_in_split_tiles(dev, heads, qo_lens, cached):
    """Values that no merge may lose or spread: V infinite or NaN for one key, a
    run of keys (several units' worth) whose scores are all -inf, K infinite for
    one key (a row that sees it is NaN)."""
    c = _Planned(dev, heads, qo_lens, cached, seed=39)
    hq, hkv, d = heads
    group, ip, ix = hq // hkv, c.csr[1].tolist(), c.csr[2].long()
    q = c.q[0].clone()
    q[..., 0] = 1.0

    def page(token):  # of the first request
        return int(ix[ip[0] + token // 16]), token % 16

    far = cached[0] - 70
    clean = c.w.run(q, c.pool).float()
    pool = c.pool.clone()
    pg, row = page(far)
    pool[pg, 1, row, 0, 3] = float("inf")
    pool[pg, 1, row, hkv - 1, 5] = float("nan")
    out = c.w.run(q, pool).float()
    n0 = qo_lens[0]
    assert bool(torch.isposinf(out[:n0, :group, 3]).all())
    assert bool(out[:n0, hq - group:, 5].isnan().all())
    out[:n0, :group, 3] = clean[:n0, :group, 3]
    out[:n0, hq - group:, 5] = clean[:n0, hq - group:, 5]
    assert torch.equal(out, clean)
    # the first 3/4 of the cached pages out of sight
    pool = c.pool.clone()
    hidden = ix[ip[0]:ip[0] + cached[0] // 16 * 3 // 4]
    pool[hidden, 0, :, :, 0] = float("-inf")
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        whole = c.w.run(q, pool)
    side.synchronize()
    out = c.w.run(q, pool)
    assert bool(out.isfinite().all()) and not torch.equal(out[:n0].float(), clean[:n0])
    # (two correct results: P is rounded to bf16 against other maxima, 2^-8 each)
    assert bool(((out.float() - whole.float()).abs() <= 2 ** -6 * whole.float().abs().clamp(min=1.0)).all())
    pool = c.pool.clone()
    pool[pg, 0, row, :, 0] = float("inf")
    out = c.w.run(q, pool)
    assert bool(out[:n0].isnan().all()) and torch.equal(out[n0:].float(), clean[n0:])
