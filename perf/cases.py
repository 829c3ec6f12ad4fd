"""The work that is timed: what a program that uses `deep_ep` has it do, through `EPBuffer` and its helpers.

A case is a dict of plain values.  Three kinds:

  serve   inference on one GPU's share: dispatch of a batch, combine of the experts' outputs.  `sync`: the host reads the
          counts (exact output sizes); without it outputs have worst-case sizes; `graph`: the two calls are captured once
          and replayed.  `payload`: 'bf16', 'fp8' (quantised on the way) or 'fp8_pair' (the caller quantises, scales come
          back as columns, as a grouped product reads them).  `biases`: rows added by the combine (a shared expert's
          output, a residual).
  train   one step's four transfers: dispatch and combine forward, the replayed dispatch of the output gradients and the
          combine of the input and gate gradients backward.
  node    all partitions of an expert-parallel group on this GPU, phase by phase: dispatch, receive, partial and final
          reduce of every partition; token counts are ragged.

`tokens` is per partition and `max_tokens` what the buffer was made for.  `zipf` 0 means near-uniform routing (the largest
of normal logits), otherwise experts have Zipf(zipf) popularity; `masked` is the share of selections that are -1.  Rows are
normal with one outlier in a thousand, padding rows are asked for as zeros, as the consumers of this layout need them.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), 'deepep-ascend_amd'))      # the package of the tree being measured

import deep_ep  # noqa: E402
from deep_ep.utils.math import per_token_cast_to_fp8  # noqa: E402

DEVICE = 'cuda'


def _case(kind, name=None, **values):
    case = dict(kind=kind, tokens=0, max_tokens=0, hidden=7168, experts=256, topk=8, alignment=128, payload='bf16', sync=True,
                graph=False, biases=0, zipf=0.0, masked=0.0, partitions=1)
    case.update(values)
    case['max_tokens'] = max(case['max_tokens'], case['tokens'])
    return case if name is None else dict(case, name=name)


def listed():
    return [
        # the smallest call that the tests and the benchmark know: a toy layer, host-synchronised, no padding
        _case('serve', 'toy_bf16', tokens=128, hidden=256, experts=8, topk=2, alignment=1),
        # decode of a small batch, replayed as a graph (no host in the loop)
        _case('serve', 'decode_graph_fp8', tokens=32, max_tokens=128, alignment=16, payload='fp8', sync=False, graph=True),
        # decode of a ragged batch, eager, without a host sync, a shared expert's output added on the way back
        _case('serve', 'decode_ragged_bf16', tokens=61, max_tokens=128, hidden=5120, experts=160, topk=6, alignment=1, sync=False,
              biases=1),
        # decode with hot and empty experts and missing selections, padded for a 128-row tile
        _case('serve', 'decode_zipf_fp8', tokens=128, payload='fp8', zipf=1.2, masked=0.1),
        # a chunk of a chunked prefill, odd sizes, an odd top-k
        _case('serve', 'chunk_ragged_bf16', tokens=1021, max_tokens=2048, hidden=2560, experts=64, topk=7, alignment=32, zipf=0.6),
        # prefill at medium size
        _case('serve', 'prefill_bf16_top8', tokens=4096),
        # prefill with rows quantised by the caller and scales returned as columns
        _case('serve', 'prefill_fp8_pair', tokens=6007, max_tokens=8192, topk=6, payload='fp8_pair'),
        # prefill at the size that the framework's benchmark quotes
        _case('serve', 'prefill_fp8_top6', tokens=16384, topk=6, payload='fp8'),
        # the largest prefill
        _case('serve', 'prefill_fp8_largest', tokens=32768, topk=8, payload='fp8'),
        # a training step's transfers
        _case('train', 'train_bf16', tokens=8192, hidden=4096, experts=128, topk=4, alignment=64),
        # decode of an expert-parallel group
        _case('node', 'node8_decode_fp8', tokens=64, max_tokens=128, alignment=16, payload='fp8', sync=False, partitions=8),
        # prefill of an expert-parallel group
        _case('node', 'node8_prefill_fp8', tokens=2048, topk=6, payload='fp8', partitions=8),
    ]


def _log_uniform(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    most = max(work(c)['bytes'] for c in listed())
    while True:
        kind = rng.choice(['serve', 'serve', 'serve', 'train', 'node'])
        # rows of 16-byte vectors; packed rows and caller-quantised ones need multiples of 32 channels
        hidden = rng.choice([256, 1024, 1536, 2048, 2560, 4096, 5120, 7168, 7168, 32 * rng.randint(8, 224)])
        experts = rng.choice([8, 32, 64, 128, 160, 256, 256, 384])
        topk = min(rng.choice([1, 2, 3, 4, 5, 6, 6, 7, 8, 8]), experts)
        alignment = rng.choice([1, 16, 32, 64, 128, 128])
        zipf = rng.choice([0.0, 0.0, 0.6, 1.2])
        masked = rng.choice([0.0, 0.0, 0.1])
        if kind == 'serve':
            tokens = _log_uniform(rng, 1, 32768)
            payload = rng.choice(['bf16', 'fp8', 'fp8', 'fp8_pair'])
            sync = tokens > 256 or rng.random() < 0.5
            case = _case(kind, tokens=tokens, max_tokens=tokens if rng.random() < 0.5 else min(32768, 2 * tokens), hidden=hidden,
                         experts=experts, topk=topk, alignment=alignment, payload=payload, sync=sync,
                         graph=not sync and rng.random() < 0.5, biases=rng.choice([0, 0, 1, 2]), zipf=zipf, masked=masked)
        elif kind == 'train':
            case = _case(kind, tokens=_log_uniform(rng, 256, 16384), hidden=hidden, experts=experts, topk=topk,
                         alignment=alignment, zipf=zipf, masked=masked)
        else:
            partitions = rng.choice([2, 4, 8])
            tokens = _log_uniform(rng, 8, 32768 // partitions)
            experts = rng.choice([64, 128, 256, 384])
            case = _case(kind, tokens=tokens, max_tokens=max(tokens, min(128, 2 * tokens)), hidden=hidden, experts=experts,
                         topk=max(2, topk), alignment=alignment, payload=rng.choice(['bf16', 'fp8', 'fp8']),
                         sync=tokens > 256, zipf=zipf, masked=masked, partitions=partitions)
        if work(case)['bytes'] <= most:
            return case


# ---- inputs ---------------------------------------------------------------------------------------

def _partition_tokens(case, rank):
    """Token counts of a group are ragged: every second partition has an eighth less."""
    return case['tokens'] if case['kind'] != 'node' else max(1, case['tokens'] - (case['tokens'] // 8 if rank % 2 else 0))


def _rows(gen, tokens, hidden):
    x = torch.randn((tokens, hidden), generator=gen, device=DEVICE)
    outlier = torch.rand((tokens, hidden), generator=gen, device=DEVICE) < 1e-3
    return torch.where(outlier, x * 50, x).to(torch.bfloat16)


def _popularity(case):
    p = np.arange(1, case['experts'] + 1, dtype=np.float64) ** -case['zipf']
    return p / p.sum()


def _routing(case, gen, rank=0):
    """Selections and gate weights of a partition's tokens.  Which experts go together is the same for every seed (the
    number of rows that a dispatch hands out depends on it); which token has which selections and which expert stands for
    which is the seed's (experts stay in their partition)."""
    tokens, experts, parts = _partition_tokens(case, rank), case['experts'], case['partitions']
    fixed = torch.Generator(device=DEVICE).manual_seed(20260 + rank)
    if case['zipf']:
        # the largest of log-popularity plus Gumbel noise: drawn without replacement
        hot = torch.randperm(experts, generator=torch.Generator(device=DEVICE).manual_seed(20259), device=DEVICE)
        u = torch.rand((tokens, experts), generator=fixed, device=DEVICE, dtype=torch.float64).clamp_(1e-12, 1 - 1e-12)
        score = torch.from_numpy(np.log(_popularity(case))).to(DEVICE)[hot] - torch.log(-torch.log(u))
    else:
        score = torch.randn((tokens, experts), generator=fixed, device=DEVICE)
    topk = torch.topk(score, case['topk'], dim=-1).indices
    missing = torch.rand((tokens, case['topk']), generator=fixed, device=DEVICE) < case['masked']
    order = torch.randperm(tokens, generator=gen, device=DEVICE)
    names = torch.rand((parts, experts // parts), generator=torch.Generator(device=DEVICE).manual_seed(gen.initial_seed() + 1),
                       device=DEVICE).argsort(dim=1)
    names = (names + torch.arange(0, experts, experts // parts, device=DEVICE)[:, None]).reshape(-1)
    topk, missing = names[topk[order]].contiguous(), missing[order]
    weights = torch.softmax(torch.randn((tokens, case['topk']), generator=gen, device=DEVICE), dim=-1)
    return (topk.masked_fill(missing, -1), weights.masked_fill(missing, 0.0)) if case['masked'] else (topk, weights)


def _expert_rows(case, topks, rank):
    """Rows that partition `rank` has after the dispatch of these selections: (received tokens, expanded rows)."""
    local = case['experts'] // case['partitions']
    received, counts = 0, np.zeros(local, dtype=np.int64)
    for topk in topks:
        e = topk.cpu().numpy()
        mine = (e >= rank * local) & (e < (rank + 1) * local)
        received += int(mine.any(axis=1).sum())
        counts += np.bincount(e[mine] - rank * local, minlength=local)
    a = case['alignment']
    return received, int(((counts + a - 1) // a * a).sum())


def _worst_rows(case):
    local, a = case['experts'] // case['partitions'], case['alignment']
    n = case['partitions'] * case['max_tokens'] * min(case['topk'], local) + (a - 1) * local
    return -(-n // a) * a


def _bf16_normal(gen, rows, hidden):
    return torch.randn((rows, hidden), generator=gen, device=DEVICE, dtype=torch.bfloat16)


def _buffer(case, group):
    return deep_ep.EPBuffer(group, num_max_tokens_per_rank=case['max_tokens'], hidden=case['hidden'], num_topk=case['topk'],
                            use_fp8_dispatch=case['payload'] != 'bf16')


def _dispatch_options(case):
    return dict(num_experts=case['experts'], num_max_tokens_per_rank=case['max_tokens'], expert_alignment=case['alignment'],
                do_expand=True, do_zero_padding=True, do_cpu_sync=case['sync'], fused_fp8_quant=case['payload'] == 'fp8')


def prepare(case, seed):
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    state = {'case': case, 'options': _dispatch_options(case)}
    if case['kind'] == 'node':
        return _prepare_node(case, gen, state)
    tokens, hidden = case['tokens'], case['hidden']
    state['x'] = _rows(gen, tokens, hidden)
    state['topk'], state['weights'] = _routing(case, gen)
    state['received'], state['expanded'] = _expert_rows(case, [state['topk']], 0)
    state['buffer'] = _buffer(case, deep_ep.LocalGroup())
    # what the experts return: as many rows as the dispatch hands out
    state['y'] = _bf16_normal(gen, state['expanded'] if case['sync'] else _worst_rows(case), hidden)
    biases = tuple(_bf16_normal(gen, tokens, hidden) for _ in range(case['biases']))
    state['bias'] = None if not biases else biases[0] if len(biases) == 1 else biases
    if case['kind'] == 'train':
        state['grad_out'] = _bf16_normal(gen, tokens, hidden)
        state['grad_rows'] = _bf16_normal(gen, state['expanded'], hidden)
        state['grad_weights'] = torch.randn((state['expanded'],), generator=gen, device=DEVICE)
    if case['graph']:
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _serve(state)
        torch.cuda.current_stream().wait_stream(side)
        state['graph'] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state['graph']):
            state['results'] = _serve(state)
    return state


def _prepare_node(case, gen, state):
    ranks = range(case['partitions'])
    node = deep_ep.LocalNode(case['partitions'])
    state['buffers'] = [_buffer(case, node.group(r)) for r in ranks]
    state['x'] = [_rows(gen, _partition_tokens(case, r), case['hidden']) for r in ranks]
    routing = [_routing(case, gen, r) for r in ranks]
    state['topk'], state['weights'] = [t for t, _ in routing], [w for _, w in routing]
    state['sizes'] = [_expert_rows(case, state['topk'], r) for r in ranks]
    state['y'] = [_bf16_normal(gen, n if case['sync'] else _worst_rows(case), case['hidden']) for _, n in state['sizes']]
    return state


# ---- one pass -------------------------------------------------------------------------------------

def _handle_outputs(handle, received):
    return [handle.psum_num_recv_tokens_per_rank, handle.psum_num_recv_tokens_per_expert,
            handle.num_unaligned_recv_tokens_per_expert, handle.dst_buffer_slot_idx, handle.recv_src_metadata[:received]]


def _serve(s):
    case = s['case']
    if case['payload'] == 'fp8_pair':
        q, scales = per_token_cast_to_fp8(s['x'])
        received, _, weights, handle, _ = s['buffer'].dispatch(
            (q, scales.view(torch.int16)), topk_idx=s['topk'], topk_weights=s['weights'], use_tma_aligned_col_major_sf=True,
            **s['options'])
    else:
        received, _, weights, handle, _ = s['buffer'].dispatch(s['x'], topk_idx=s['topk'], topk_weights=s['weights'],
                                                               **s['options'])
    out, out_weights, _ = s['buffer'].combine(s['y'], handle, topk_weights=weights, bias=s['bias'])
    # (without a host sync the tensors are longer than what was written: the rest is not looked at)
    n = s['expanded']
    rows, sf = received if isinstance(received, tuple) else (received, None)
    return [rows[:n], None if sf is None else sf[:n], weights[:n], out, out_weights, *_handle_outputs(handle, s['received'])]


def _train(s):
    buffer = s['buffer']
    rows, _, weights, handle, _ = buffer.dispatch(s['x'], topk_idx=s['topk'], topk_weights=s['weights'], **s['options'])
    out, out_weights, _ = buffer.combine(s['y'], handle, topk_weights=weights)
    grad_y, _, _, _, _ = buffer.dispatch(s['grad_out'], handle=handle, do_expand=True, do_zero_padding=True)
    grad_x, grad_gate, _ = buffer.combine(s['grad_rows'], handle, topk_weights=s['grad_weights'])
    return [rows, weights, out, out_weights, grad_y, grad_x, grad_gate, *_handle_outputs(handle, s['received'])]


def _node(s):
    deferred = dict(async_with_compute_stream=True, defer_epilogue=True)
    sent = [b.dispatch(x, topk_idx=t, topk_weights=w, **deferred, **s['options'])
            for b, x, t, w in zip(s['buffers'], s['x'], s['topk'], s['weights'])]
    got = [event.current_stream_wait() for event in sent]
    reduced = [b.combine(y, handle, topk_weights=weights, **deferred)
               for b, y, (_, _, weights, handle) in zip(s['buffers'], s['y'], got)]
    results = [event.current_stream_wait() for event in reduced]
    outputs = []
    for (rows, _, weights, handle), (out, out_weights), (received, n) in zip(got, results, s['sizes']):
        parts = rows if isinstance(rows, tuple) else (rows,)
        outputs.append([*(p[:n] for p in parts), weights[:n], out, out_weights, handle.psum_num_recv_tokens_per_expert,
                        handle.dst_buffer_slot_idx, handle.recv_src_metadata[:received]])
    return outputs


def run(state):
    if state['case']['kind'] == 'node':
        return _node(state)
    if state['case']['kind'] == 'train':
        return _train(state)
    if state['case']['graph']:
        state['graph'].replay()
        return state['results']
    return _serve(state)


# ---- bytes and tolerance -----------------------------------------------------------------------------

def _expected_padding(case, tokens):
    """Padding rows of all partitions: the mean of (-count) modulo the alignment over Poisson counts."""
    a = case['alignment']
    if a == 1:
        return 0.0
    mean = tokens * case['topk'] * (1 - case['masked'])
    # (drawing without replacement caps an expert at one row a token)
    lam = np.minimum(mean * (_popularity(case) if case['zipf'] else np.full(case['experts'], 1 / case['experts'])), tokens)
    total = 0.0
    for x in lam if case['zipf'] else lam[:1]:
        if x > 8 * a:
            pad = (a - 1) / 2
        else:
            c = np.arange(0, int(x + 12 * math.sqrt(x) + 12))
            log_p = c * math.log(max(x, 1e-300)) - x - np.cumsum(np.log(np.maximum(c, 1)))
            pad = float((np.exp(log_p) * (-c % a)).sum())
        total += pad * (1 if case['zipf'] else case['experts'])
    return total


def work(case):
    h, k, r = case['hidden'], case['topk'], case['partitions']
    tokens = sum(_partition_tokens(case, p) for p in range(r))
    valid = tokens * k * (1 - case['masked'])
    padding = _expected_padding(case, tokens)
    groups = -(-h // 128)
    row = (h + 4 * groups if case['payload'] != 'bf16' else 2 * h) + 4           # payload, scales, gate weight
    metadata = tokens * (k + 2) * 4
    into = tokens * (2 * h + k * (8 + 4 + 4)) + (valid + padding) * row + metadata
    back = valid * (2 * h + 4) + tokens * 2 * h * (1 + case['biases']) + tokens * k * (4 + 8) + metadata
    flops = valid * h
    total = into + back
    if case['payload'] == 'fp8_pair':
        total += tokens * (h + 4 * groups) * 2 - tokens * h                       # quantised rows written, then read
    if case['payload'] != 'bf16':
        flops += 3 * tokens * h
    if case['kind'] == 'train':
        total += tokens * 2 * h + (valid + padding) * 2 * h + metadata + back
        flops *= 2
    if case['kind'] == 'node':
        # a token is packed once for every partition that it goes to, and comes back as one partial of each
        local = case['experts'] // r
        hit = 1 - (1 - local / case['experts']) ** (k * (1 - case['masked']))
        packed = tokens * r * hit
        total += packed * (2 * (row + 12 * k) + 2 * 2 * h)
    return {'bytes': float(total), 'flops': float(flops)}


def tolerance(case):
    # Copies, quantised bytes, scales, weights and indices are exact.  Combined rows are float32 sums of at most ten bfloat16
    # terms rounded once (twice with biases): summed in the opposite order a few in ten million land on the other side of a
    # rounding boundary (measured: rel 1.2e-6, single values 5e-3 away); one such value is 3e-5 of the smallest case's output.
    return {'rel': 1e-4, 'max': 0.02}
