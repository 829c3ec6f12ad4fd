"""Dispatches of decode size, layout and copy in one launch: handles and rows of the oracle at the edges of what that
launch takes, in every payload form, with and without a host sync, and the calls around it that it must not change."""
import ctypes

import numpy as np
import pytest
import torch

from helpers import bf16_bits, make_routing, make_tokens
from oracle import ep_oracle as O

pytestmark = pytest.mark.gpu
DEV = 'cuda'

CASES = [
    # T, H, E, K, A, masked, zipf
    (1, 128, 1, 1, 1, 0.0, None),
    (1, 16, 40, 32, 3, 0.2, None),
    (32, 128, 2048, 32, 1, 0.1, None),      # every entry of the limit, the largest expert count
    (33, 128, 64, 32, 4, 0.0, None),        # one entry row beyond it: two launches
    (128, 528, 24, 8, 128, 0.3, None),      # every entry of the limit, both sides of a 512-channel part
    (128, 1040, 256, 8, 16, 0.1, 1.2),      # hot and empty experts
    (127, 2064, 8, 3, 8, 0.5, None),
    (129, 256, 16, 2, 64, 0.0, None),       # one token beyond it
    (64, 256, 300, 16, 1, 0.0, None),       # more experts than threads
    (128, 64, 2048, 1, 16, 0.0, None),      # more pieces of padding (4096) than workgroups that zero them (1024)
    (128, 2080, 160, 8, 128, 0.0, None),    # the same with more than 48 MiB of padding in BF16 (2560 pieces, 2048 workgroups)
]


@pytest.mark.parametrize('T,H,E,K,A,masked,zipf', CASES)
@pytest.mark.parametrize('mode', ['bf16', 'fused', 'pair'])
def test_small_dispatch(T, H, E, K, A, masked, zipf, mode):
    import deep_ep
    x = make_tokens(T, H, seed=T + H, outliers=True)
    topk, w = make_routing(T, E, K, seed=T + K, masked=masked, zipf=zipf)
    if T > 2 and K > 1:
        topk[2], w[2] = -1, 0.0             # a token that nobody receives
        topk[0, 1] = topk[0, 0]             # an expert selected twice
    lay = O.rank_share_layout(topk.numpy(), E, 1, 0, A, T)
    n, ne = lay['num_recv_tokens'], lay['num_expanded_tokens']
    buf = deep_ep.EPBuffer(deep_ep.LocalGroup(), num_max_tokens_per_rank=T + 5, hidden=H, num_topk=K, use_fp8_dispatch=mode != 'bf16',
                           explicitly_destroy=True)
    q, s = O.quantise(x)
    xin = x.to(DEV) if mode != 'pair' else (q.view(torch.float8_e4m3fn).to(DEV), s.view(torch.int16).to(DEV))
    ex, es, ew = O.rank_share_dispatch(bf16_bits(x) if mode == 'bf16' else q.numpy(), None if mode == 'bf16' else s.numpy().view(np.uint32),
                                       w.numpy(), lay)
    stats = torch.zeros(E, dtype=torch.int32, device=DEV)
    for k, sync in enumerate((True, False, True)):
        recv, _, rw, handle, _ = buf.dispatch(xin, topk_idx=topk.to(DEV), topk_weights=w.to(DEV), num_experts=E,
                                              num_max_tokens_per_rank=T + 5, expert_alignment=A, do_expand=True, do_zero_padding=True,
                                              do_cpu_sync=sync, fused_fp8_quant=mode == 'fused', cumulative_local_expert_recv_stats=stats)
        torch.cuda.synchronize()
        for name in ('psum_num_recv_tokens_per_rank', 'psum_num_recv_tokens_per_expert', 'num_unaligned_recv_tokens_per_expert',
                     'dst_buffer_slot_idx', 'dst_gsge_idx'):
            assert np.array_equal(getattr(handle, name).cpu().numpy(), lay[name]), name
        meta = lay['recv_src_metadata'].copy()
        assert np.array_equal(handle.recv_src_metadata.cpu().numpy()[:n], meta)
        assert np.array_equal(stats.cpu().numpy(), (k + 1) * lay['num_unaligned_recv_tokens_per_expert'])
        if sync:
            assert handle.num_recv_tokens == n and handle.num_expanded_tokens == ne
            assert handle.num_recv_tokens_per_expert_list == lay['num_recv_tokens_per_expert_list']
        rows, sf = recv if isinstance(recv, tuple) else (recv, None)
        got = bf16_bits(rows) if mode == 'bf16' else rows.view(torch.uint8).cpu().numpy()
        assert np.array_equal(got[:ne], ex)
        if sf is not None:
            assert np.array_equal(np.ascontiguousarray(sf.cpu().numpy()).view(np.uint32).reshape(sf.size(0), -1)[:ne], es)
        assert np.array_equal(rw.cpu().numpy().view(np.uint32)[:ne], ew.view(np.uint32))
    buf.destroy()


@pytest.mark.parametrize('T,E,K,A,masked', [(1, 8, 8, 1, 0.0), (32, 9, 3, 4, 0.3), (33, 255, 8, 1, 0.0), (64, 1024, 16, 128, 0.0),
                                            (65, 1025, 15, 3, 0.1), (96, 4, 4, 7, 0.0), (128, 1024, 8, 1, 0.2), (128, 2048, 8, 96, 0.0)])
@pytest.mark.parametrize('R', [1, 2])
def test_small_dispatch_each_expert_once(T, E, K, A, masked, R):
    """No token selects an expert twice: ranks are counted in the bits of the tokens below (up to 1024 experts), at the edges of
    the words that hold them and of the groups of experts that are scanned."""
    import deep_ep
    H, E = 64, E + E % R
    x = [make_tokens(T, H, seed=T + r) for r in range(R)]
    rt = [make_routing(T, E, K, seed=T + K + r, masked=masked) for r in range(R)]
    assert all(len(set(row[row >= 0])) == (row >= 0).sum() for topk, _ in rt for row in topk.numpy())
    node = deep_ep.LocalNode(R) if R > 1 else None
    bufs = [deep_ep.EPBuffer(node.group(r) if R > 1 else deep_ep.LocalGroup(), num_max_tokens_per_rank=T, hidden=H, num_topk=K,
                             explicitly_destroy=True) for r in range(R)]
    args = dict(num_experts=E, num_max_tokens_per_rank=T, expert_alignment=A, do_expand=True, do_zero_padding=True, do_cpu_sync=False)
    if R == 1:
        got = [bufs[0].dispatch(x[0].to(DEV), topk_idx=rt[0][0].to(DEV), topk_weights=rt[0][1].to(DEV), **args)]
    else:
        events = [b.dispatch(xx.to(DEV), topk_idx=t.to(DEV), topk_weights=w.to(DEV), async_with_compute_stream=True, defer_epilogue=True, **args)
                  for b, xx, (t, w) in zip(bufs, x, rt)]
        got = [e.current_stream_wait() for e in events]
    torch.cuda.synchronize()
    El = E // R
    for r in range(R):
        rows, _, weights, handle = got[r][:4]
        # the stable order: sources in turn, their tokens ascending, positions ascending inside a token
        entries = [[] for _ in range(El)]
        for s in range(R):
            for t in range(T):
                for j in range(K):
                    e = int(rt[s][0][t, j]) - r * El
                    if 0 <= e < El:
                        entries[e].append((s, t, j))
        assert [len(e) for e in entries] == handle.num_unaligned_recv_tokens_per_expert.cpu().tolist()
        start, want, want_w = 0, [], []
        rows, weights = bf16_bits(rows), weights.cpu().numpy()
        for e in entries:
            for i, (s, t, j) in enumerate(e):
                want.append((start + i, bf16_bits(x[s])[t]))
                want_w.append((start + i, rt[s][1][t, j].item()))
            n = -(-len(e) // A) * A
            assert not rows[start + len(e):start + n].any() and not weights[start + len(e):start + n].any()
            start += n
        at = [i for i, _ in want]
        assert np.array_equal(rows[at], np.stack([v for _, v in want])) and np.array_equal(weights[at], np.float32([v for _, v in want_w]))
        masters = (rt[r][0].numpy() >= 0) & (rt[r][0].numpy() < E)
        slots = handle.dst_buffer_slot_idx.cpu().numpy()
        for p in range(R):          # a token's last selection of a partition has its place among the tokens that go there
            seen = 0
            for t in range(T):
                js = [j for j in range(K) if masters[t, j] and int(rt[r][0][t, j]) // El == p]
                assert all(slots[t, j] == -1 for j in js[:-1])
                if js:
                    assert slots[t, js[-1]] == seen
                    seen += 1
    for b in bufs:
        b.destroy()


CHUNK_CASES = [
    # T, H, E, K, A, masked, zipf
    (130, 16, 8, 1, 1, 0.0, None),          # one workgroup a wave's worth of tasks each
    (200, 512, 2048, 32, 16, 0.1, None),    # most experts, most entries a token, 16 own tokens a workgroup (one part a row)
    (512, 528, 40, 32, 3, 0.3, None),       # every entry of the limit
    (2048, 272, 256, 8, 128, 0.1, 1.2),     # the same, hot and empty experts
    (4096, 64, 5, 4, 64, 0.5, None),        # and every token
    (1021, 2576, 64, 7, 32, 0.0, None),     # tokens shared by two workgroups
    (300, 5136, 300, 5, 16, 0.2, None),     # two workgroups a CU
    (1366, 64, 12, 12, 1, 0.0, None),       # beyond the entries: two launches
    (4097, 64, 8, 2, 8, 0.0, None),         # beyond the tokens
]


@pytest.mark.parametrize('T,H,E,K,A,masked,zipf', CHUNK_CASES)
@pytest.mark.parametrize('mode', ['bf16', 'fused', 'pair'])
def test_chunk_dispatch(T, H, E, K, A, masked, zipf, mode):
    """The same of dispatches beyond decode size that are one launch, at the edges of what that takes."""
    test_small_dispatch(T, H, E, K, A, masked, zipf, mode)


def test_small_dispatch_deferred_exact_and_replayed():
    """The same handles from the calls that keep the two launches (a deferred epilogue, exact sizes), and a cached
    dispatch behind the single launch."""
    import deep_ep
    T, H, E, K, A = 50, 256, 16, 4, 8
    x = make_tokens(T, H, seed=1).to(DEV)
    topk, w = make_routing(T, E, K, seed=2, masked=0.2)
    args = dict(topk_idx=topk.to(DEV), topk_weights=w.to(DEV), num_experts=E, num_max_tokens_per_rank=T, expert_alignment=A,
                do_expand=True, do_zero_padding=True)
    buf = deep_ep.EPBuffer(deep_ep.LocalGroup(), num_max_tokens_per_rank=T, hidden=H, num_topk=K, explicitly_destroy=True)
    r0, _, w0, h0, _ = buf.dispatch(x, **args)
    deferred = buf.dispatch(x, async_with_compute_stream=True, defer_epilogue=True, **args)
    r1, _, w1, h1 = deferred.current_stream_wait()
    buf.set_exact_sync_sizes(True)
    r2, _, w2, h2, _ = buf.dispatch(x, **args)
    buf.set_exact_sync_sizes(False)
    r3, _, w3, _, _ = buf.dispatch(x, topk_weights=w.to(DEV), handle=h0, do_expand=True, do_zero_padding=True)
    torch.cuda.synchronize()
    for r, ww, h in ((r1, w1, h1), (r2, w2, h2), (r3, w3, h0)):
        assert torch.equal(r.view(torch.int16), r0.view(torch.int16)) and torch.equal(ww, w0)
        assert torch.equal(h.recv_src_metadata, h0.recv_src_metadata)
        assert torch.equal(h.dst_buffer_slot_idx, h0.dst_buffer_slot_idx)
    buf.destroy()


@pytest.mark.parametrize('T,E,K', [(1021, 64, 7), (1024, 256, 8), (1025, 256, 8), (257, 48, 21), (900, 16, 6), (8192, 8, 1), (2048, 32, 2),
                                   (2049, 32, 2), (1281, 64, 5), (256, 256, 8), (257, 256, 8), (512, 64, 4), (513, 64, 4), (2048, 8, 1),
                                   (2049, 8, 1), (2048, 64, 3), (2049, 64, 3), (1536, 64, 4), (1537, 64, 4), (768, 256, 8), (769, 256, 8), (512, 16, 8),
                                   (513, 16, 8), (640, 32, 6), (641, 32, 6), (257, 32, 7), (1024, 8, 4), (1025, 8, 4), (512, 33, 4), (513, 33, 4),
                                   (512, 64, 16), (513, 64, 16)])
def test_ids_of_all_blocks_counted_in_place(T, E, K):
    """Around the most blocks x top-k (64) for which the histogram kernel can be left out (every workgroup then reads all ids
    itself), and around the library's own limits: 16 (of few experts, up to 32 for top-6: 32) without and 48 with a host that waits, 16 blocks, and 64 where the layout
    does not rank in bit masks (top-16).  The same handles whichever launches run.  (The layout has launches of its own where
    the epilogue is deferred, and beyond 4096 tokens or 16384 entries.)"""
    import deep_ep
    H, A = 64, 4
    x = make_tokens(T, H, seed=T).to(DEV)
    topk, w = make_routing(T, E, K, seed=K, masked=0.1)
    topk[5] = -1
    lay = O.rank_share_layout(topk.numpy(), E, 1, 0, A, T)
    buf = deep_ep.EPBuffer(deep_ep.LocalGroup(), num_max_tokens_per_rank=T, hidden=H, num_topk=K, explicitly_destroy=True)
    try:
        for limit, sync in ((64, True), (-1, True), (-1, False)):
            deep_ep._C.set_layout_recount_limit(limit)
            args = dict(topk_idx=topk.to(DEV), num_experts=E, expert_alignment=A, do_expand=True, do_cpu_sync=sync)
            handles = [buf.dispatch(x, **args)[3],
                       buf.dispatch(x, async_with_compute_stream=True, defer_epilogue=True, **args).current_stream_wait()[3]]
            torch.cuda.synchronize()
            for handle in handles:
                for name in ('psum_num_recv_tokens_per_rank', 'psum_num_recv_tokens_per_expert', 'num_unaligned_recv_tokens_per_expert',
                             'dst_buffer_slot_idx'):
                    assert np.array_equal(getattr(handle, name).cpu().numpy(), lay[name]), (limit, sync, name)
                assert np.array_equal(handle.recv_src_metadata.cpu().numpy()[:lay['num_recv_tokens']], lay['recv_src_metadata'])
                if sync:
                    assert handle.num_recv_tokens_per_expert_list == lay['num_recv_tokens_per_expert_list']
    finally:
        deep_ep._C.set_layout_recount_limit(-1)
    buf.destroy()


@pytest.mark.parametrize('T,E,K,how', [(2049, 9, 7, ''), (1153, 256, 8, ''), (3001, 1024, 8, ''), (20001, 8, 1, ''), (4224, 130, 3, ''), (2100, 256, 8, 'twice'),
                                       (1400, 8, 8, 'one'), (2305, 257, 5, 'few'), (3000, 1025, 8, ''), (2200, 64, 9, '')])
def test_slots_from_bits(T, E, K, how):
    """The two layout launches of one partition that rank in bit masks (up to top-8 and 1024 experts; the last two cases are beyond), at
    the edges of blocks, words and groups of experts, in more count rows than one go holds (3001 tokens, 1024 experts), with
    experts selected twice (every entry on one expert: the most passes), and with most selections missing."""
    import deep_ep
    H, A = 16, 4
    x = make_tokens(T, H, seed=T).to(DEV)
    topk, _ = make_routing(T, E, K, seed=K, masked=0.95 if how == 'few' else 0.1)
    if how == 'twice':
        topk[::3, K - 1] = topk[::3, 0]
        topk[1::7, 2] = topk[1::7, 1]
    if how == 'one':
        topk[:] = 3
    topk[130] = -1
    topk[T - 1, :] = E + 1                      # (no such expert)
    lay = O.rank_share_layout(np.where(topk.numpy() < E, topk.numpy(), -1), E, 1, 0, A, T)
    buf = deep_ep.EPBuffer(deep_ep.LocalGroup(), num_max_tokens_per_rank=T, hidden=H, num_topk=K, explicitly_destroy=True)
    try:
        deep_ep._C.set_layout_recount_limit(0)
        handle = buf.dispatch(x, topk_idx=topk.to(DEV), num_experts=E, expert_alignment=A, do_expand=True, async_with_compute_stream=True,
                              defer_epilogue=True).current_stream_wait()[3]
        torch.cuda.synchronize()
    finally:
        deep_ep._C.set_layout_recount_limit(-1)
    for name in ('psum_num_recv_tokens_per_rank', 'psum_num_recv_tokens_per_expert', 'num_unaligned_recv_tokens_per_expert',
                 'dst_buffer_slot_idx', 'recv_src_metadata'):
        assert np.array_equal(getattr(handle, name).cpu().numpy(), lay[name]), name
    assert handle.num_recv_tokens_per_expert_list == lay['num_recv_tokens_per_expert_list']
    buf.destroy()


def _repeated(T, E, K, how, seed):
    """Selections in which tokens select an expert more than once."""
    g = torch.Generator().manual_seed(seed)
    topk = torch.randint(0, E, (T, K), generator=g)
    if how == 'stairs':                         # 1, 2, .. K times, at any place of the token, beside distinct ones
        topk, _ = make_routing(T, E, K, seed=seed)
        for t in range(T):
            topk[t, torch.randperm(K, generator=g)[:t % K + 1]] = topk[t, 0].item()
    if how == 'last':                           # the last token's last two entries and no other
        topk, _ = make_routing(T, E, K, seed=seed)
        topk[T - 1, K - 1] = topk[T - 1, K - 2]
    if how == 'same':                           # all of a token, the first and the last expert most
        topk = torch.tensor([0, E - 1, E // 2])[torch.randint(0, 3, (T, 1), generator=g)].expand(T, K).contiguous()
    return topk


@pytest.mark.parametrize('T,E,K,how', [(1153, 8, 8, 'any'), (200, 9, 8, 'any'), (2049, 64, 8, 'stairs'), (1400, 1024, 7, 'stairs'), (1283, 256, 5, 'stairs'),
                                       (1793, 256, 8, 'last'), (3000, 32, 2, 'last'), (2177, 1024, 8, 'same'), (1500, 48, 3, 'same'), (4100, 8, 4, 'any')])
@pytest.mark.parametrize('masked', [False, True])
def test_slots_from_bits_of_repeated_selections(T, E, K, how, masked):
    """The second, third, .. selections of an expert by a token leave their bits a pass each: up to top-k passes, an entry alone in the
    last one, missing selections in between."""
    import deep_ep
    H, A = 16, 4
    x = make_tokens(T, H, seed=T).to(DEV)
    topk = _repeated(T, E, K, how, seed=T + K)
    if masked:
        topk[torch.rand((T, K), generator=torch.Generator().manual_seed(3)) < 0.2] = -1
    lay = O.rank_share_layout(topk.numpy(), E, 1, 0, A, T)
    buf = deep_ep.EPBuffer(deep_ep.LocalGroup(), num_max_tokens_per_rank=T, hidden=H, num_topk=K, explicitly_destroy=True)
    try:
        deep_ep._C.set_layout_recount_limit(0)
        handle = buf.dispatch(x, topk_idx=topk.to(DEV), num_experts=E, expert_alignment=A, do_expand=True, async_with_compute_stream=True,
                              defer_epilogue=True).current_stream_wait()[3]
        torch.cuda.synchronize()
    finally:
        deep_ep._C.set_layout_recount_limit(-1)
    for name in ('psum_num_recv_tokens_per_rank', 'psum_num_recv_tokens_per_expert', 'num_unaligned_recv_tokens_per_expert',
                 'dst_buffer_slot_idx', 'recv_src_metadata'):
        assert np.array_equal(getattr(handle, name).cpu().numpy(), lay[name]), name
    buf.destroy()


@pytest.mark.parametrize('T,E,K,how', [(128, 16, 8, 'stairs'), (128, 1024, 8, 'same'), (127, 256, 8, 'stairs'), (65, 64, 3, 'any'), (17, 1025, 5, 'stairs'),
                                       (2, 24, 8, 'same'), (1, 16, 8, 'same'), (31, 64, 32, 'stairs'), (128, 160, 6, 'last')])
@pytest.mark.parametrize('R', [1, 2])
def test_small_dispatch_of_repeated_selections(T, E, K, how, R):
    """Decode sizes: none, a wave's worth (64) and many more entries beyond the first of a token for an expert, in the order of sources,
    tokens and positions (1025 experts: without masks)."""
    import deep_ep
    H, A, El = 32, 4, (E + E % R) // R
    x = [make_tokens(T, H, seed=T + r).to(DEV) for r in range(R)]
    topk = [_repeated(T, E, K, how, seed=T + K + r) for r in range(R)]
    gates = [torch.rand((T, K), generator=torch.Generator().manual_seed(r)) for r in range(R)]
    node = deep_ep.LocalNode(R) if R > 1 else None
    bufs = [deep_ep.EPBuffer(node.group(r) if R > 1 else deep_ep.LocalGroup(), num_max_tokens_per_rank=T, hidden=H, num_topk=K,
                             explicitly_destroy=True) for r in range(R)]
    args = dict(num_experts=El * R, num_max_tokens_per_rank=T, expert_alignment=A, do_expand=True, do_cpu_sync=False)
    if R == 1:
        got = [bufs[0].dispatch(x[0], topk_idx=topk[0].to(DEV), topk_weights=gates[0].to(DEV), **args)]
    else:
        events = [b.dispatch(xx, topk_idx=t.to(DEV), topk_weights=g.to(DEV), async_with_compute_stream=True, defer_epilogue=True, **args)
                  for b, xx, t, g in zip(bufs, x, topk, gates)]
        got = [e.current_stream_wait() for e in events]
    torch.cuda.synchronize()
    every = torch.cat([t.reshape(-1) for t in topk])
    rows_of = torch.cat([xx.cpu().repeat_interleave(K, dim=0) for xx in x])
    gate_of = torch.cat([g.reshape(-1) for g in gates])
    for r in range(R):
        rows, _, weights, handle = got[r][:4]
        local = torch.where((every >= r * El) & (every < (r + 1) * El), every - r * El, El)
        counts = torch.bincount(local, minlength=El + 1)[:El]
        assert torch.equal(handle.num_unaligned_recv_tokens_per_expert.cpu().long(), counts)
        order = torch.argsort(local, stable=True)[:int(counts.sum())]
        aligned = (counts + A - 1) // A * A
        starts = torch.cumsum(aligned, 0) - aligned
        slots = starts[local[order]] + torch.arange(len(order)) - (torch.cumsum(counts, 0) - counts)[local[order]]
        assert torch.equal(rows.cpu()[slots].view(torch.int16), rows_of[order].view(torch.int16))
        assert torch.equal(weights.cpu()[slots], gate_of[order])
    for b in bufs:
        b.destroy()


def test_a_layout_of_repeated_selections_takes_no_multiple_of_one_without():
    """A layout of several blocks behind the histograms, timed as replays of a captured graph: every selection of a token on one expert costs
    up to seven passes over a block's masks (half as much again), not a look through all of its repetitions (eight times)."""
    import deep_ep
    T, H, E, K, calls = 4096, 16, 256, 8, 8
    buf = deep_ep.EPBuffer(deep_ep.LocalGroup(), num_max_tokens_per_rank=T, hidden=H, num_topk=K, explicitly_destroy=True)
    x = make_tokens(T, H).to(DEV)
    distinct, _ = make_routing(T, E, K, seed=1)

    def shortest(topk):
        topk = topk.to(DEV)

        def dispatches():
            return [buf.dispatch(x, topk_idx=topk, num_experts=E, num_max_tokens_per_rank=T, expert_alignment=1, do_expand=True, do_cpu_sync=False,
                                 async_with_compute_stream=True, defer_epilogue=True) for _ in range(calls)]
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            dispatches()
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            kept = dispatches()
        times = []
        for _ in range(20):
            begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            begin.record()
            graph.replay()
            end.record()
            end.synchronize()
            times.append(begin.elapsed_time(end))
        del kept
        return min(times)

    assert shortest(distinct[:, :1].expand(T, K).contiguous()) < 3 * shortest(distinct)
    buf.destroy()


class AbiDispatch:
    """One BF16 dispatch through the C ABI: descriptors and outputs of the two calls it is made of."""

    def __init__(self, C, buf, T, H, E, K, A, x, topk, w):
        n_recv, n_exp = ctypes.c_int(), ctypes.c_int()
        C._check(C._ep_worst(None, T, K, E, A, ctypes.byref(n_recv), ctypes.byref(n_exp)))
        i32 = dict(dtype=torch.int32, device=DEV)
        self.C, self.buf = C, buf
        self.keep = (x, topk, w)
        self.psum_expert = torch.full((E,), -7, **i32)
        self.counts = [torch.full((1,), -7, **i32), torch.full((E,), -7, **i32), torch.full((T, K), -7, **i32)]
        self.dst_slot = torch.full((T, K), -7, **i32)
        self.meta = torch.full((T, K + 2), -7, **i32)
        self.rows = torch.full((n_exp.value, H), 77, dtype=torch.int16, device=DEV).view(torch.bfloat16)
        self.gates = torch.full((n_exp.value,), -7.0, device=DEV)
        self.a, self.e = C._DispatchArgs(), C._DispatchEpilogueArgs()
        for f in (self.a, self.e):
            f.x, f.topk_weights = C._desc(x), C._desc(w)
            f.psum_num_recv_tokens_per_rank, f.psum_num_recv_tokens_per_expert = C._desc(self.counts[0]), C._desc(self.psum_expert)
            f.num_max_tokens_per_rank, f.num_experts, f.expert_alignment = T, E, A
        self.a.topk_idx, self.a.num_unaligned_recv_tokens_per_expert = C._desc(topk), C._desc(self.counts[1])
        self.a.dst_buffer_slot_idx, self.a.dst_gsge_idx = C._desc(self.dst_slot), C._desc(self.counts[2])
        self.e.recv_x, self.e.recv_topk_weights, self.e.recv_src_metadata = C._desc(self.rows), C._desc(self.gates), C._desc(self.meta)
        self.e.num_topk, self.e.do_zero_padding = K, 1
        torch.cuda.synchronize()

    def begin(self, stream, call='begin'):
        self.a.stream = stream.cuda_stream
        begin = {'begin': self.C._ep_dispatch_begin, 'begin_only': self.C._ep_dispatch_begin_only}[call]
        self.C._check(begin(self.buf.runtime._h, ctypes.byref(self.a)))
        self.e.dispatch_stamp = self.C._ep_stamp(self.buf.runtime._h)

    def epilogue(self, stream):
        self.e.stream = stream.cuda_stream
        self.C._check(self.C._ep_dispatch_epi(self.buf.runtime._h, ctypes.byref(self.e)))

    def check(self, x, topk, w, E, A):
        T = x.size(0)
        lay = O.rank_share_layout(topk.numpy(), E, 1, 0, A, T)
        n, ne = lay['num_recv_tokens'], lay['num_expanded_tokens']
        ex, _, ew = O.rank_share_dispatch(bf16_bits(x), None, w.numpy(), lay)
        assert np.array_equal(self.psum_expert.cpu().numpy(), lay['psum_num_recv_tokens_per_expert'])
        assert np.array_equal(self.dst_slot.cpu().numpy(), lay['dst_buffer_slot_idx'])
        assert np.array_equal(self.meta.cpu().numpy()[:n], lay['recv_src_metadata'])
        assert np.array_equal(bf16_bits(self.rows)[:ne], ex)
        assert np.array_equal(self.gates.cpu().numpy().view(np.uint32)[:ne], ew.view(np.uint32))


BEGINS = [(96, 'begin'), (64, 'begin_only'), (700, 'begin_only'), (4096, 'begin_only')]       # the last two in a launch of chunk size


@pytest.mark.parametrize('T,call', BEGINS)
def test_begin_and_epilogue_on_two_streams(T, call):
    """The epilogue of an ep_dispatch_begin on another stream, ordered behind the begin by an event only: the ids arrive
    late on the first stream, and every pass routes differently, so that a layout of the pass before would show."""
    import deep_ep
    C = deep_ep._C
    H, E, K, A = 256, 16, 4, 8
    buf = deep_ep.EPBuffer(deep_ep.LocalGroup(), num_max_tokens_per_rank=T, hidden=H, num_topk=K, explicitly_destroy=True)
    x = make_tokens(T, H, seed=4)
    first, second = torch.cuda.Stream(), torch.cuda.Stream()
    for seed in range(4):
        topk, w = make_routing(T, E, K, seed=20 + seed, masked=0.1 * seed)
        source, late = topk.to(DEV), torch.full_like(topk, -1).to(DEV)
        d = AbiDispatch(C, buf, T, H, E, K, A, x.to(DEV), late, w.to(DEV))
        with torch.cuda.stream(first):
            for _ in range(4):
                junk = torch.randn((1024, 1024), device=DEV) @ torch.randn((1024, 1024), device=DEV)
            late.copy_(source)
        d.begin(first, call)
        second.wait_event(first.record_event())
        d.epilogue(second)
        torch.cuda.synchronize()
        del junk
        d.check(x, topk, w, E, A)
    buf.destroy()


@pytest.mark.parametrize('T,call', BEGINS)
def test_cached_epilogue_between_begin_and_its_epilogue(T, call):
    """A replay of another handle between the two calls leaves the waiting layout where it is."""
    import deep_ep
    C = deep_ep._C
    H, E, K, A = 256, 16, 4, 8
    buf = deep_ep.EPBuffer(deep_ep.LocalGroup(), num_max_tokens_per_rank=T, hidden=H, num_topk=K, explicitly_destroy=True)
    x = make_tokens(T, H, seed=6)
    stream = torch.cuda.current_stream()
    old_topk, old_w = make_routing(T, E, K, seed=40)
    old = AbiDispatch(C, buf, T, H, E, K, A, x.to(DEV), old_topk.to(DEV), old_w.to(DEV))
    old.begin(stream, call)
    old.epilogue(stream)
    topk, w = make_routing(T, E, K, seed=41, masked=0.2)
    d = AbiDispatch(C, buf, T, H, E, K, A, x.to(DEV), topk.to(DEV), w.to(DEV))
    d.begin(stream, call)
    old.rows.zero_()
    old.e.cached_mode = 1
    old.epilogue(stream)
    d.epilogue(stream)
    torch.cuda.synchronize()
    old.check(x, old_topk, old_w, E, A)
    d.check(x, topk, w, E, A)
    with pytest.raises(C.EPException, match='one copy epilogue'):
        d.epilogue(stream)
    buf.destroy()


@pytest.mark.parametrize('T', [129, 700, 2049])
def test_begin_beyond_decode_size_enqueues_its_layout(T):
    """What an ep_dispatch_begin of more than 128 tokens serves: the ids may change behind it on its stream, the counts can be
    waited for before the epilogue, and epilogues may come again, padded otherwise too."""
    import deep_ep
    C = deep_ep._C
    H, E, K, A = 128, 16, 4, 8
    buf = deep_ep.EPBuffer(deep_ep.LocalGroup(), num_max_tokens_per_rank=T, hidden=H, num_topk=K, explicitly_destroy=True)
    x = make_tokens(T, H, seed=9)
    topk, w = make_routing(T, E, K, seed=44, masked=0.2)
    lay = O.rank_share_layout(topk.numpy(), E, 1, 0, A, T)
    ids = topk.to(DEV)
    d = AbiDispatch(C, buf, T, H, E, K, A, x.to(DEV), ids, w.to(DEV))
    d.a.do_cpu_sync = 1
    stream = torch.cuda.current_stream()
    d.begin(stream)
    ids.fill_(-1)
    n, ne, per_expert = ctypes.c_int(), ctypes.c_int(), (ctypes.c_int * E)()
    C._check(C._ep_wait(buf.runtime._h, ctypes.byref(n), ctypes.byref(ne), per_expert))
    assert (n.value, ne.value) == (lay['num_recv_tokens'], lay['num_expanded_tokens'])
    assert list(per_expert) == lay['num_recv_tokens_per_expert_list']
    d.epilogue(stream)
    torch.cuda.synchronize()
    d.check(x, topk, w, E, A)
    d.rows.view(torch.int16).fill_(77)
    d.e.expert_alignment = 1
    d.epilogue(stream)
    torch.cuda.synchronize()
    slots = lay['recv_src_metadata'][:, :K]
    real = np.zeros(ne.value, dtype=bool)
    real[slots[slots >= 0]] = True
    rows, ex = bf16_bits(d.rows)[:ne.value], O.rank_share_dispatch(bf16_bits(x), None, w.numpy(), lay)[0]
    assert np.array_equal(rows[real], ex[real]) and (rows[~real].view(np.int16) == 77).all() and not real.all()
    d.e.expert_alignment = A
    d.epilogue(stream)
    torch.cuda.synchronize()
    d.check(x, topk, w, E, A)
    buf.destroy()


@pytest.mark.parametrize('T,call', BEGINS)
@pytest.mark.parametrize('field,value', [('experts', 64), ('experts', 8), ('alignment', 16)])
def test_epilogue_of_other_experts_or_alignment_is_refused(field, value, T, call):
    """The one launch counts in LDS sized by the begin's experts: an epilogue that names others is refused on the host,
    and the right one still runs; so is a wait for the counts in between."""
    import deep_ep
    C = deep_ep._C
    H, E, K, A = 128, 16, 4, 8
    buf = deep_ep.EPBuffer(deep_ep.LocalGroup(), num_max_tokens_per_rank=T, hidden=H, num_topk=K, explicitly_destroy=True)
    x = make_tokens(T, H, seed=7)
    topk, w = make_routing(T, E, K, seed=42, masked=0.2)
    d = AbiDispatch(C, buf, T, H, E, K, A, x.to(DEV), topk.to(DEV), w.to(DEV))
    stream = torch.cuda.current_stream()
    d.begin(stream, call)
    with pytest.raises(C.EPException, match='comes before the counts'):
        C._check(C._ep_wait(buf.runtime._h, None, None, None))
    if field == 'experts':
        other = torch.zeros(value, dtype=torch.int32, device=DEV)
        d.e.num_experts, d.e.psum_num_recv_tokens_per_expert = value, C._desc(other)
    else:
        d.e.expert_alignment = value
    with pytest.raises(C.EPException, match='of its ep_dispatch_begin'):
        d.epilogue(stream)
    d.e.num_experts, d.e.expert_alignment, d.e.psum_num_recv_tokens_per_expert = E, A, C._desc(d.psum_expert)
    d.epilogue(stream)
    torch.cuda.synchronize()
    d.check(x, topk, w, E, A)
    buf.destroy()


@pytest.mark.parametrize('T', [64, 129])
def test_static_dispatch_with_an_epilogue_of_its_own_alignment(T):
    """The static entry point takes an epilogue that pads to another alignment than its layout's, at any size: the rows are
    those of the layout, and alignment 1 leaves the padding as it was."""
    import deep_ep
    C = deep_ep._C
    H, E, K, A = 128, 16, 4, 8
    buf = deep_ep.EPBuffer(deep_ep.LocalGroup(), num_max_tokens_per_rank=T, hidden=H, num_topk=K, explicitly_destroy=True)
    x = make_tokens(T, H, seed=8)
    topk, w = make_routing(T, E, K, seed=43, masked=0.2)
    d = AbiDispatch(C, buf, T, H, E, K, A, x.to(DEV), topk.to(DEV), w.to(DEV))
    d.e.expert_alignment = 1
    d.a.stream = d.e.stream = torch.cuda.current_stream().cuda_stream
    C._check(C._ep_dispatch_static(ctypes.byref(d.a), ctypes.byref(d.e)))
    torch.cuda.synchronize()
    lay = O.rank_share_layout(topk.numpy(), E, 1, 0, A, T)
    n, ne = lay['num_recv_tokens'], lay['num_expanded_tokens']
    ex, _, _ = O.rank_share_dispatch(bf16_bits(x), None, w.numpy(), lay)
    assert np.array_equal(d.meta.cpu().numpy()[:n], lay['recv_src_metadata'])
    slots = lay['recv_src_metadata'][:, :K]
    real = np.zeros(ne, dtype=bool)
    real[slots[slots >= 0]] = True
    rows = bf16_bits(d.rows)[:ne]
    assert np.array_equal(rows[real], ex[real]) and (rows[~real].view(np.int16) == 77).all() and not real.all()
    buf.destroy()
