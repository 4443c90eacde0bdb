"""The calls a user of this framework makes, with the sizes they make them at: single decode steps of the three
operators and of the kernels in front of them, from one token or request to the largest batch, and MoE prefill.

Everything goes through ``cuda_agent_amd.capi``. A case is a dict of plain values; ``path`` names the chain:

  gdn     one decode step of a Gated DeltaNet layer: ``plain`` is the recurrence alone, ``layer`` the causal
          convolution update followed by the recurrence with its pre-step and the gated norm of the read-out
  attend  sparse-MLA attention over rows that are already selected
  sparse  the whole sparse attention step: indexer scores, top-k selection, attention over the selected rows
  moe     the FP8 MoE layer from router logits to the combined output
  router  what stands in front of the MoE layer: RMS norm with quantiser, router projection, routing
"""

import math

import torch

from __graft_entry__ import load_package

load_package()

from cuda_agent_amd import capi  # noqa: E402

PAGE = 64


def _gdn(batch, heads=32, qk_heads=16, dtype='bf16', form='layer'):
    return dict(path='gdn', batch=batch, heads=heads, qk_heads=qk_heads, dtype=dtype, form=form)


def _attend(batch, rows, topk=2048, heads=128, cache='bf16', paged=False):
    return dict(path='attend', batch=batch, heads=heads, rows=rows, topk=topk, cache=cache, paged=paged)


def _sparse(batch, rows, topk=2048, heads=128, cache='bf16', paged=False, ragged=False):
    return dict(path='sparse', batch=batch, heads=heads, rows=rows, topk=topk, cache=cache, paged=paged,
                ragged=ragged)


def _moe(tokens, hidden=7168, inter=2048, experts=256, top_k=8, biased=False, shared=False, pow2=False):
    return dict(path='moe', tokens=tokens, hidden=hidden, inter=inter, experts=experts, top_k=top_k, biased=biased,
                shared=shared, pow2=pow2)


def _router(tokens, hidden=7168, experts=256, top_k=8, split=True):
    return dict(path='router', tokens=tokens, hidden=hidden, experts=experts, top_k=top_k, split=split)


def listed():
    return [
        # one request of a small recurrent layer, fp32 throughout: the latency of a single launch
        dict(_gdn(1, 16, 16, 'fp32', 'plain'), name='gdn_single'),
        # a serving batch of odd size through everything a layer does between its projections
        dict(_gdn(37), name='gdn_layer_37'),
        # a full serving batch: 537 MB of state read and written
        dict(_gdn(256, form='plain'), name='gdn_batch_256'),
        # one request over a long context: the latency of a token for an interactive user
        dict(_sparse(1, 65536), name='sparse_single'),
        # a ragged batch over a paged cache in its 8-bit form, the way a server with a full card keeps it
        dict(_sparse(24, 33000, cache='e4m3', paged=True, ragged=True), name='sparse_paged_24'),
        # attention alone at the size of a full decode batch
        dict(_attend(64, 32768), name='attend_64'),
        # one token through the MoE layer (interactive decode)
        dict(_moe(1), name='moe_single'),
        # a decode batch: nearly every expert's weights are streamed for one or two tokens each
        dict(_moe(64), name='moe_decode_64'),
        # a chunk of a prompt (or a very large decode batch) with a shared expert on every token
        dict(_moe(1500, shared=True), name='moe_chunk_1500'),
        # a long prompt with skewed expert load
        dict(_moe(8192, biased=True), name='moe_prefill_8192'),
        # norm, router projection and routing of a decode batch: four small launches
        dict(_router(64), name='router_decode_64'),
        # the same for a long prompt
        dict(_router(8192), name='router_prefill_8192'),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    path = rng.choice(['gdn', 'attend', 'sparse', 'moe', 'moe', 'router'])
    if path == 'gdn':
        heads, qk_heads = rng.choice([(16, 16), (32, 16), (32, 32), (8, 4), (48, 16)])
        return _gdn(_log_int(rng, 1, 8192 // heads), heads, qk_heads, rng.choice(['bf16', 'bf16', 'fp32']),
                    rng.choice(['plain', 'layer']))
    if path in ('attend', 'sparse'):
        # (at most the 2 million cached positions of 64 requests x 32768)
        batch = _log_int(rng, 1, 200)
        rows = _log_int(rng, 3000, min(131072, (64 * 32768) // batch))
        cache = rng.choice(['bf16', 'bf16', 'e4m3'])
        heads = rng.choice([128, 128, 128, 64, 32])
        topk = rng.choice([2048, 2048, 1024, 512, rng.randint(64, 2048)])
        paged = rng.random() < 0.5
        if path == 'attend':
            return _attend(batch, rows, topk, heads, cache, paged)
        return _sparse(batch, rows, topk, heads, cache, paged, rng.random() < 0.5)
    if path == 'moe':
        hidden, inter, experts, top_k = rng.choice([(7168, 2048, 256, 8), (7168, 2048, 256, 8), (2048, 768, 128, 8),
                                                    (4096, 1536, 64, 4)])
        shared = rng.random() < 0.3
        return _moe(_log_int(rng, 1, 4096 if shared else 8192), hidden, inter, experts, top_k, rng.random() < 0.3,
                    shared, rng.random() < 0.25)
    hidden = rng.choice([7168, 7168, 2048, 4096])
    return _router(_log_int(rng, 1, 8192), hidden, rng.choice([256, 256, 128, 64]), 8, rng.random() < 0.7)


# ---- inputs ------------------------------------------------------------------------------------------------

def _rng(seed):
    return torch.Generator(device='cuda').manual_seed(seed)


def _randn(gen, *shape):
    return torch.randn(*shape, device='cuda', generator=gen)


def _rand(gen, *shape):
    return torch.rand(*shape, device='cuda', generator=gen)


def _prepare_gdn(case, gen):
    B, Hv, Hqk = case['batch'], case['heads'], case['qk_heads']
    dt = torch.bfloat16 if case['dtype'] == 'bf16' else torch.float32
    s = {'state': 0.02 * _randn(gen, B, Hv, 128, 128)}
    q, k = _randn(gen, B, Hqk, 128), _randn(gen, B, Hqk, 128)
    if case['form'] == 'plain':
        s['q'] = (q / q.norm(dim=-1, keepdim=True)).to(dt)
        s['k'] = (k / k.norm(dim=-1, keepdim=True)).to(dt)
        s['v'] = _randn(gen, B, Hv, 128).to(dt)
        s['g'] = torch.exp(-0.5 * torch.nn.functional.softplus(_randn(gen, B, Hv)))
        s['beta'] = torch.sigmoid(_randn(gen, B, Hv))
        s['out'] = torch.empty(B, Hv, 128, device='cuda')
        return s
    channels = (2 * Hqk + Hv) * 128
    s['x'] = _randn(gen, B, channels).to(dt)
    s['conv_state'] = _randn(gen, B, channels, 4).to(dt)
    s['weight'] = (0.5 * _randn(gen, channels, 4)).to(dt)
    s['bias'] = (0.1 * _randn(gen, channels)).to(dt)
    s['a'], s['b'] = _randn(gen, B, Hv), _randn(gen, B, Hv)
    s['a_log'] = torch.log(1.0 + 15.0 * _rand(gen, Hv))
    s['dt_bias'] = 0.5 * _randn(gen, Hv)
    s['z'] = _randn(gen, B, Hv, 128).to(dt)
    s['norm_w'] = (1.0 + 0.1 * _randn(gen, 128)).to(dt)
    s['q'] = torch.empty(B, Hqk * 128, device='cuda', dtype=dt)
    s['k'] = torch.empty(B, Hqk * 128, device='cuda', dtype=dt)
    s['v'] = torch.empty(B, Hv * 128, device='cuda', dtype=dt)
    s['out'] = torch.empty(B, Hv, 128, device='cuda', dtype=dt)
    return s


def _run_gdn(case, s):
    B, Hv, Hqk = case['batch'], case['heads'], case['qk_heads']
    if case['form'] == 'plain':
        capi.gdn_decode_launch(s['out'], s['state'], s['q'], s['k'], s['v'], s['g'], s['beta'])
        return s['out'], s['state']
    capi.causal_conv1d_update_launch(s['q'], s['k'], s['v'], s['conv_state'], s['x'], s['weight'], s['bias'])
    capi.gdn_decode_fused_norm_launch(s['out'], s['state'], s['q'].view(B, Hqk, 128), s['k'].view(B, Hqk, 128),
                                      s['v'].view(B, Hv, 128), s['a'], s['b'], s['a_log'], s['dt_bias'], s['z'],
                                      s['norm_w'])
    return s['out'], s['state'], s['conv_state']


def _cache_rows(case):
    """Rows of the cache block of one request (whole pages when it is paged)."""
    return -(-case['rows'] // PAGE) * PAGE if case['paged'] else case['rows']


def _prepare_attend(case, gen):
    B, H, k = case['batch'], case['heads'], case['topk']
    N = _cache_rows(case)
    e4m3 = case['cache'] == 'e4m3'
    s = {'q': _randn(gen, B, H, 576).bfloat16()}
    if e4m3:
        s['kv'] = torch.empty(B, N, capi.LATENT_ROW_BYTES, dtype=torch.uint8, device='cuda')
    else:
        s['kv'] = torch.empty(B, N, 576, dtype=torch.bfloat16, device='cuda')
    for b in range(B):
        rows = _randn(gen, N, 576).bfloat16()
        if e4m3:
            capi.mla_latent_quant_launch(s['kv'][b], rows)
        else:
            s['kv'][b] = rows
    if case['paged']:
        s['kv'] = s['kv'].view(B * N // PAGE, PAGE, -1)
        s['table'] = torch.randperm(B * N // PAGE, device='cuda', generator=gen).int().view(B, N // PAGE)
    s['out'] = torch.empty(B, H, 512, dtype=torch.bfloat16, device='cuda')
    size = capi.sparse_mla_fp8_workspace_bytes if e4m3 else capi.sparse_mla_workspace_bytes
    s['workspace'] = torch.empty(size(B, H, k), dtype=torch.uint8, device='cuda')
    if case['path'] == 'attend':
        picked = torch.stack([torch.randperm(case['rows'], device='cuda', generator=gen)[:k] for _ in range(B)])
        if picked.shape[1] < k:  # fewer rows than asked for: the rest is padding
            picked = torch.nn.functional.pad(picked, (0, k - picked.shape[1]), value=-1)
        s['idx'] = picked.int().contiguous()
    return s


def _run_attend(case, s):
    if case['cache'] == 'e4m3':
        if case['paged']:
            capi.sparse_mla_decode_fp8_paged_launch(s['out'], s['q'], s['kv'], s['table'], s['idx'], s['workspace'])
        else:
            capi.sparse_mla_decode_fp8_launch(s['out'], s['q'], s['kv'], s['idx'], s['workspace'])
    elif case['paged']:
        capi.sparse_mla_decode_paged_launch(s['out'], s['q'], s['kv'], s['table'], s['idx'], s['workspace'])
    else:
        capi.sparse_mla_decode_launch(s['out'], s['q'], s['kv'], s['idx'], s['workspace'])
    return s['out']


def _prepare_sparse(case, gen):
    s = _prepare_attend(case, gen)
    B, N = case['batch'], _cache_rows(case)
    keys = _randn(gen, B, N, 128)
    query = _randn(gen, B, 64, 128)
    s['index_w'] = _randn(gen, B, 64) / 8
    if case['cache'] == 'e4m3':
        # codes and one scale per row, as the activation quantiser writes them; the query's scales go into the weights
        s['keys'] = torch.empty(B * N, 128, dtype=torch.uint8, device='cuda')
        s['key_scale'] = torch.empty(B * N, 1, device='cuda')
        capi.moe_quant_bf16_launch(s['keys'], s['key_scale'], keys.bfloat16().view(B * N, 128))
        codes, scales = torch.empty(B * 64, 128, dtype=torch.uint8, device='cuda'), torch.empty(B * 64, 1, device='cuda')
        capi.moe_quant_bf16_launch(codes, scales, query.bfloat16().view(B * 64, 128))
        s['index_q'] = codes.view(B, 64, 128)
        s['index_w'] = (s['index_w'] * scales.view(B, 64)).contiguous()
        shape = (B * N // PAGE, PAGE) if case['paged'] else (B, N)
        s['keys'], s['key_scale'] = s['keys'].view(*shape, 128), s['key_scale'].view(*shape)
    else:
        s['keys'], s['index_q'] = keys.bfloat16(), query.bfloat16()
        if case['paged']:
            s['keys'] = s['keys'].view(B * N // PAGE, PAGE, 128)
    rows = case['rows']
    if case['ragged']:
        s['lengths'] = torch.randint(max(1, rows // 4), rows + 1, (B,), device='cuda', generator=gen, dtype=torch.int32)
    else:
        s['lengths'] = torch.full((B,), rows, dtype=torch.int32, device='cuda')
    s['scores'] = torch.empty(B, N, device='cuda')
    s['idx'] = torch.empty(B, case['topk'], dtype=torch.int32, device='cuda')
    return s


def _run_sparse(case, s):
    args = (s['index_w'], s['lengths'])
    if case['cache'] == 'e4m3':
        if case['paged']:
            capi.mla_index_scores_fp8_paged_launch(s['scores'], s['index_q'], s['keys'], s['key_scale'], s['table'], *args)
        else:
            capi.mla_index_scores_fp8_launch(s['scores'], s['index_q'], s['keys'], s['key_scale'], *args)
    elif case['paged']:
        capi.mla_index_scores_paged_launch(s['scores'], s['index_q'], s['keys'], s['table'], *args)
    else:
        capi.mla_index_scores_launch(s['scores'], s['index_q'], s['keys'], *args)
    capi.topk_select_launch(s['idx'], s['scores'], s['lengths'])
    return s['scores'], s['idx'], _run_attend(case, s)


def _codes(gen, experts, rows, cols):
    """Expert weights N(0, 1/cols) as e4m3 codes of 448 times that, a few experts at a time."""
    out = torch.empty(experts, rows, cols, dtype=torch.float8_e4m3fn, device='cuda')
    step = max(1, (1 << 28) // (rows * cols))
    for e in range(0, experts, step):
        n = min(step, experts - e)
        out[e:e + n] = (_randn(gen, n, rows, cols) * (448 / cols ** 0.5)).to(torch.float8_e4m3fn)
    return out


def _prepare_moe(case, gen):
    T, H, I, E, k = (case[n] for n in ('tokens', 'hidden', 'inter', 'experts', 'top_k'))
    stored = E + (1 if case['shared'] else 0)
    s = {'x': _randn(gen, T, H).bfloat16(), 'logits': _randn(gen, T, E)}
    if case['biased']:
        s['logits'][:, torch.randperm(E, device='cuda', generator=gen)[:E // 16]] += 2.0
    s['w13'], s['w2'] = _codes(gen, stored, 2 * I, H), _codes(gen, stored, H, I)
    s['w13_s'] = (0.5 + _rand(gen, stored, 2 * I // 128, H // 128)) / 448
    s['w2_s'] = (0.5 + _rand(gen, stored, H // 128, I // 128)) / 448
    if case['pow2']:
        for name in ('w13_s', 'w2_s'):
            s[name] = torch.exp2(torch.ceil(torch.log2(s[name])))
    size = capi.moe_workspace_bytes(T, H, I, stored, k + stored - E)
    s['workspace'] = torch.empty(size, dtype=torch.uint8, device='cuda')
    s['out'] = torch.empty(T, H, dtype=torch.bfloat16, device='cuda')
    return s


def _run_moe(case, s):
    launch = capi.moe_fp8_fused_shared_launch if case['shared'] else capi.moe_fp8_launch
    launch(s['out'], s['x'], s['logits'], s['w13'], s['w13_s'], s['w2'], s['w2_s'], s['workspace'],
           top_k=case['top_k'], config=capi.CONFIG_UE8M0 if case['pow2'] else 0)
    return s['out']


def _prepare_router(case, gen):
    T, H, E, k = (case[n] for n in ('tokens', 'hidden', 'experts', 'top_k'))
    s = {'x': _randn(gen, T, H).bfloat16(), 'norm_w': (1.0 + 0.1 * _randn(gen, H)).bfloat16(),
         'weight': _randn(gen, E, H) * H ** -0.5, 'bias': 0.1 * _randn(gen, E)}
    if case['split']:
        s['planes'] = torch.empty(3, E, H, dtype=torch.bfloat16, device='cuda')
        capi.moe_router_split_weight_launch(s['planes'], s['weight'])
    s['y'] = torch.empty(T, H, dtype=torch.bfloat16, device='cuda')
    s['codes'] = torch.empty(T, H, dtype=torch.uint8, device='cuda')
    s['scales'] = torch.empty(T, H // 128, device='cuda')
    s['logits'] = torch.empty(T, E, device='cuda')
    s['ids'] = torch.empty(T, k, dtype=torch.int32, device='cuda')
    s['weights'] = torch.empty(T, k, device='cuda')
    size = capi.moe_router_logits_workspace_bytes(T, H, E)
    s['workspace'] = torch.empty(size, dtype=torch.uint8, device='cuda') if size else None
    return s


def _run_router(case, s):
    capi.moe_rmsnorm_quant_launch(s['codes'], s['scales'], s['y'], s['x'], s['norm_w'])
    if case['split']:
        capi.moe_router_logits_split_launch(s['logits'], s['y'], s['planes'], s['workspace'])
    else:
        capi.moe_router_logits_launch(s['logits'], s['y'], s['weight'], s['workspace'])
    capi.moe_route_grouped_launch(s['ids'], s['weights'], s['logits'], s['bias'], 8, 4, True, 2.5)
    return s['y'], s['codes'], s['scales'], s['logits'], s['ids'], s['weights']


_PREPARE = dict(gdn=_prepare_gdn, attend=_prepare_attend, sparse=_prepare_sparse, moe=_prepare_moe, router=_prepare_router)
_RUN = dict(gdn=_run_gdn, attend=_run_attend, sparse=_run_sparse, moe=_run_moe, router=_run_router)


def prepare(case, seed):
    return case, _PREPARE[case['path']](case, _rng(seed))


def run(state):
    case, tensors = state
    return _RUN[case['path']](case, tensors)


# ---- the work of one pass, and what two correct evaluations may differ by -------------------------------------

def work(case):
    path = case['path']
    if path == 'gdn':
        B, Hv, Hqk = case['batch'], case['heads'], case['qk_heads']
        e = 2 if case['dtype'] == 'bf16' else 4
        vectors = B * (2 * Hqk + Hv) * 128
        bytes_ = 2 * B * Hv * 128 * 128 * 4 + 2 * B * Hv * 4
        flops = B * Hv * 128 * 128 * 7
        if case['form'] == 'plain':
            return dict(bytes=bytes_ + vectors * e + B * Hv * 128 * 4, flops=flops)
        channels = (2 * Hqk + Hv) * 128
        return dict(bytes=bytes_ + vectors * e * 9 + channels * 5 * e + 2 * B * Hv * 128 * e, flops=flops + 8 * vectors)
    if path in ('attend', 'sparse'):
        B, H, rows, k = case['batch'], case['heads'], case['rows'], min(case['topk'], case['rows'])
        e4m3 = case['cache'] == 'e4m3'
        bytes_ = B * k * (656 if e4m3 else 1152) + B * H * (576 + 512) * 2 + B * case['topk'] * 4
        flops = 2 * B * H * k * (576 + 512)
        if path == 'sparse':
            # ragged lengths are uniform between a quarter of the rows and all of them
            live = int(rows * 0.625) if case['ragged'] else rows
            bytes_ += B * live * (128 + 4 if e4m3 else 256) + B * _cache_rows(case) * 4 + B * case['topk'] * 4
            bytes_ += B * 64 * 128 * (1 if e4m3 else 2)
            flops += 2 * B * 64 * live * 128
        return dict(bytes=bytes_, flops=flops)
    if path == 'moe':
        T, H, I, E, k = (case[n] for n in ('tokens', 'hidden', 'inter', 'experts', 'top_k'))
        # experts that at least one of T tokens routes to, if the choices are even
        active = E * (1 - (1 - k / E) ** T) + (1 if case['shared'] else 0)
        expert = 3 * I * H + 3 * I * H // 128 // 128 * 4
        return dict(bytes=int(active * expert) + 2 * T * H * 2 + T * E * 4,
                    flops=6 * T * (k + (1 if case['shared'] else 0)) * H * I)
    T, H, E, k = (case[n] for n in ('tokens', 'hidden', 'experts', 'top_k'))
    return dict(bytes=T * H * 5 + T * (H // 128) * 4 + 2 * H + E * H * (6 if case['split'] else 4) + T * E * 4 + T * k * 8,
                flops=2 * T * H * E)


def tolerance(case):
    path = case['path']
    if path == 'gdn':
        if case['form'] == 'plain' or case['dtype'] == 'fp32':
            # fp32 sums: 8e-8 off a float64 evaluation (largest 5e-7), three passes deep at most
            return dict(rel=2e-6, max=1e-5)
        return dict(rel=6e-3, max=3e-2)  # the read-out in bf16: one rounding step is 2^-8 of a value
    if path == 'attend':
        # split counts against each other: 2.0e-3, largest 8.4e-3 (bf16 probabilities and output)
        return dict(rel=8e-3, max=3.4e-2)
    if path == 'sparse':
        # as above. The selection of float64 scores was the same in 24 of 24 rows; a row whose last place is
        # decided by the order of fp32 sums would list its entries shifted by one
        return dict(rel=8e-3, max=3.4e-2, differ=1e-2)
    if path == 'moe':
        # the layer's forms (streaming or tiled, bf16 or e4m3 matrix core) against each other: 1.9e-3, largest
        # 4.9e-2: a code of the requantised intermediate that fp32 does not decide moves single outputs that far
        return dict(rel=8e-3, max=0.2)
    # 3e-5 of the normalised values land on the neighbouring bf16 value of a float64 evaluation (rel 3.3e-5); the
    # projection is 2e-7 off one
    return dict(rel=1e-3, max=3.4e-2, differ=1e-3)
