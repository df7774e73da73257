"""The work that this framework's performance is measured on.

A case is a plain dict; `listed()` gives the fixed ones and `draw(rng)` further ones of the same ranges. `prepare`
makes what a user's program holds before the call (inputs on the GPU, caches, weights, the engine), `run` makes one
pass through the public entry points, `work` counts the bytes and operations the pass cannot do without, `tolerance`
says how far another correct implementation may be, and `exact` gives the result in 64 bits from plain torch.
"""
import math
import random

import torch

from streamvoxel_amd import synth
from streamvoxel_amd.stream.attention import attention
from streamvoxel_amd.stream.backbone import run_block
from streamvoxel_amd.stream.engine import Encoded, SlotEngine
from streamvoxel_amd.stream.forward import GatherPatch
from streamvoxel_amd.stream.patches import PatchLogits
from streamvoxel_amd.stream.step import CachedContext, EaseSelect

DEVICE = 'cuda'


def listed():
    return [
        # One cross-attention layer of the 8-slot step: 12 x 64 heads, every window's own count of cached keys
        # (1552 of the wide and biome context, 1024 more for each neighbour that exists).
        _attend('context_8_windows', windows=8, heads=12, head_dim=64, low=1552, high=9744, grain=1024, pick=11),
        # The same layer for the one window that a lone player's column waits for, all eight neighbours there.
        _attend('context_1_window', windows=1, heads=12, head_dim=64, low=9744, high=9744, grain=1024, pick=1),
        # The shipped model's cross-attention: 8 x 48 heads, 4096 prefix keys and 288 + 1024 k local ones.
        _attend('context_shipped', windows=8, heads=8, head_dim=48, low=4384, high=12576, grain=1024, pick=7),
        # Many players on one card, their context held in e4m3 to fit: 64 windows, 16 x 64 heads.
        _attend('context_64_windows_e4m3', windows=64, heads=16, head_dim=64, low=1552, high=9744, grain=1024, pick=5,
                cache='fp8'),
        # The masked attention of a batch padded to its longest prefix and its longest local part: a hole in the
        # middle of every shorter window's keys.
        _masked('masked_4_windows', windows=4, heads=12, head_dim=64, prefix=4096, local=5632, dtype='bf16', pick=3),
        # The single-column configuration, which keeps fp32 from end to end.
        _masked('single_column_fp32', windows=1, heads=12, head_dim=64, prefix=0, local=9744, dtype='fp32', pick=2),
        # One window's condition taken into a layer's cache when its slot is loaded: prefix rows and local keys.
        dict(name='load_window', kind='write', heads=8, head_dim=48, prefix=4096, local=8480, capacity=12672,
             cache='bf16'),
        # One backbone block of the shipped model over the 8 slots (1024 patch tokens each).
        dict(name='block_8_windows', kind='block', windows=8, tokens=1024, width=768, timed=True),
        # The embedding of the 8 slots' voxels, half of them still masked.
        dict(name='patchify_8_windows', kind='patchify', windows=8, height=256, width=768, classes=304, masked=0.5),
        # The selection of a solid step over the class head's rows where they lie (shipped model, 8 slots).
        dict(name='select_8_windows', kind='select', windows=8, height=256, classes=304, dtype='bf16', layout='patch',
             done=0.5, peaked=0.8),
        # The same for one window whose logits come as [C, Y, Z, X] planes, as the reference's forward returns them.
        dict(name='select_1_window', kind='select', windows=1, height=256, classes=256, dtype='fp32', layout='planes',
             done=0.2, peaked=0.7),
        # A whole forward of the shipped model through the slot engine: 8 slots, 25 backbone and 13 control blocks.
        dict(name='step_8_slots', kind='step', windows=8, low=4384, high=12576, grain=1024, pick=7),
    ]


def draw(rng):
    kind = rng.choice(['attend', 'attend', 'masked', 'fp32', 'write', 'block', 'patchify', 'select', 'select', 'step'])
    pick = rng.randrange(1 << 20)
    if kind == 'attend':
        case = _attend(None, windows=_log(rng, 1, 32), heads=rng.choice([4, 8, 12, 16]),
                       head_dim=rng.choice([48, 64, 64, 96]), low=64, high=_log(rng, 256, 12576), grain=1, pick=pick,
                       cache=rng.choice(['bf16', 'bf16', 'fp8']), queries=rng.choice([1024, _log(rng, 64, 1024)]))
        case['low'] = rng.randint(1, case['high'])
        return case
    if kind == 'masked':
        return _masked(None, windows=_log(rng, 1, 8), heads=rng.choice([8, 12]), head_dim=rng.choice([48, 64, 96]),
                       prefix=_log(rng, 64, 4096), local=_log(rng, 64, 8480), dtype='bf16', pick=pick)
    if kind == 'fp32':
        return _masked(None, windows=_log(rng, 1, 4), heads=rng.choice([8, 12]), head_dim=rng.choice([48, 64]),
                       prefix=rng.choice([0, _log(rng, 64, 1024)]), local=_log(rng, 128, 8192), dtype='fp32',
                       pick=pick)
    if kind == 'write':
        prefix, local = rng.choice([0, _log(rng, 16, 4096)]), _log(rng, 16, 8480)
        return dict(kind='write', heads=rng.choice([8, 16]), head_dim=rng.choice([48, 96]), prefix=prefix, local=local,
                    capacity=prefix + local + rng.randint(0, 4096), cache=rng.choice(['bf16', 'fp8']))
    if kind == 'block':
        return dict(kind='block', windows=_log(rng, 1, 12), tokens=rng.choice([1024, _log(rng, 100, 1024)]),
                    width=rng.choice([384, 768]), timed=rng.random() < 0.7)
    if kind == 'patchify':
        return dict(kind='patchify', windows=_log(rng, 1, 16), height=16 * rng.randint(1, 16),
                    width=rng.choice([384, 768]), classes=rng.choice([256, 304]), masked=round(rng.random(), 2))
    if kind == 'select':
        return dict(kind='select', windows=_log(rng, 1, 16), height=rng.choice([64, 128, 256]),
                    classes=rng.choice([256, 304, 8 * rng.randint(2, 40)]), dtype=rng.choice(['fp32', 'bf16']),
                    layout=rng.choice(['patch', 'voxels', 'planes']), done=round(0.9 * rng.random(), 2),
                    peaked=round(rng.uniform(0.6, 0.95), 2))
    return dict(kind='step', windows=rng.randint(1, 8), low=4384, high=4384 + 1024 * rng.randint(0, 8),
                grain=rng.choice([1, 1024]), pick=pick)


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _attend(name, windows, heads, head_dim, low, high, grain, pick, cache='bf16', queries=1024):
    case = dict(kind='attend', windows=windows, heads=heads, head_dim=head_dim, queries=queries, low=low, high=high,
                grain=grain, pick=pick, cache=cache)
    return case if name is None else dict(name=name, **case)


def _masked(name, windows, heads, head_dim, prefix, local, dtype, pick, queries=1024):
    case = dict(kind='masked', windows=windows, heads=heads, head_dim=head_dim, queries=queries, prefix=prefix,
                local=local, dtype=dtype, pick=pick)
    return case if name is None else dict(name=name, **case)


def _lengths(case):
    """Each window's count of keys; the longest possible one is there."""
    rng = random.Random(case['pick'])
    steps = (case['high'] - case['low']) // case['grain']
    lengths = [case['low'] + case['grain'] * rng.randint(0, steps) for _ in range(case['windows'])]
    lengths[rng.randrange(len(lengths))] = case['low'] + case['grain'] * steps
    return lengths


def _valid(case):
    """The (prefix, local) key counts of every window of a masked batch; one window fills each part."""
    rng = random.Random(case['pick'])
    n = case['windows']
    prefix = [rng.randint(case['prefix'] // 4, case['prefix']) for _ in range(n)]
    local = [rng.randint(max(1, case['local'] // 8), case['local']) for _ in range(n)]
    prefix[rng.randrange(n)], local[rng.randrange(n)] = case['prefix'], case['local']
    return list(zip(prefix, local))


def _generator(seed):
    return torch.Generator(DEVICE).manual_seed(seed)


def _normal(g, *shape, dtype=torch.bfloat16):
    return torch.randn(*shape, device=DEVICE, generator=g).to(dtype)


# ------------------------------------------------------------------------------------------------------- inputs

def _attend_inputs(case, seed):
    g = _generator(seed)
    H, D = case['heads'], case['head_dim']
    query = _normal(g, case['windows'], case['queries'], H, D)
    return query, [(_normal(g, H, L, D), _normal(g, H, L, D)) for L in _lengths(case)]


def _masked_inputs(case, seed):
    g = _generator(seed)
    B, H, D, keys = case['windows'], case['heads'], case['head_dim'], case['prefix'] + case['local']
    dtype = torch.float32 if case['dtype'] == 'fp32' else torch.bfloat16
    query = _normal(g, B, H, case['queries'], D, dtype=dtype)
    key, value = _normal(g, B, H, keys, D, dtype=dtype), _normal(g, B, H, keys, D, dtype=dtype)
    mask = torch.zeros(B, keys, dtype=torch.bool)
    for b, (prefix, local) in enumerate(_valid(case)):
        mask[b, :prefix] = True
        mask[b, case['prefix']:case['prefix'] + local] = True
    return query, key, value, mask.to(DEVICE)


def _write_inputs(case, seed):
    g = _generator(seed)
    H, D, P, L = case['heads'], case['head_dim'], case['prefix'], case['local']
    kv = _normal(g, L, 2, H, D)          # the layer's key_value projection of the local context
    positions = torch.rand(L, 3, device=DEVICE, generator=g) * 64 - 8
    prefix = (_normal(g, H, P, D), _normal(g, H, P, D)) if P else None
    return kv, positions, prefix


def _frequencies(head_dim):
    axis = head_dim // 3
    return (10000.0 ** (-torch.arange(0, axis, 2).float() / axis)).to(DEVICE)


def _block_inputs(case, seed):
    g = _generator(seed)
    block = synth.BlockWeights(case['width'], 8, timed=case['timed'], seed=seed)
    for p in block.parameters():
        p.data = p.data.to(torch.bfloat16)
    block = block.to(DEVICE)
    n, N, W = case['windows'], case['tokens'], case['width']
    positions = synth.patch_positions().to(DEVICE)[None, :N].expand(n, -1, -1)
    return block, _normal(g, n, N, W), _normal(g, n, W) if case['timed'] else None, positions


def _world(g, shape, classes, masked):
    """Voxels of half-finished windows: a masked share, air for half of the rest, then ever rarer classes."""
    u = torch.rand(shape, device=DEVICE, generator=g)
    rare = (torch.exp(u * math.log(classes)) - 1).long().clamp_(0, classes - 1)
    air = torch.rand(shape, device=DEVICE, generator=g) < 0.5
    tokens = torch.where(air, torch.zeros_like(rare), rare)
    hidden = torch.rand(shape, device=DEVICE, generator=g) < masked
    return torch.where(hidden, torch.full_like(tokens, classes), tokens)


def _patchify_inputs(case, seed):
    g = _generator(seed)
    W, C = case['width'], case['classes']
    conv = torch.nn.Module()
    conv.weight = torch.nn.Parameter(torch.randn(W, C + 1, 4, 4, 4, device=DEVICE, generator=g) * 0.05)
    conv.bias = torch.nn.Parameter(torch.randn(W, device=DEVICE, generator=g) * 0.02)
    return conv, _world(g, (case['windows'], case['height'], 16, 16), C, case['masked'])


def _select_inputs(case, seed):
    """Logits and the state of windows in the middle of their generation."""
    g = _generator(seed)
    B, C, shape = case['windows'], case['classes'], (case['height'], 16, 16)
    N = shape[0] * 256
    dtype = torch.float32 if case['dtype'] == 'fp32' else torch.bfloat16
    logits = synth.bimodal_logits_(torch.empty(B * N, C, device=DEVICE), case['peaked'], generator=g)
    logits = logits.to(dtype).view(B, N, C)
    top = torch.randint(shape[0] // 2, shape[0] + 1, (B, 1, 16, 16), device=DEVICE, generator=g)
    last = (torch.arange(shape[0], device=DEVICE)[None, :, None, None] >= top).reshape(B, N)
    # Every block has had its share of the steps so far, to a voxel: the quota keeps them in step.
    split = lambda x: x.view(B, shape[0] // 4, 4, 4, 4, 4, 4).permute(0, 1, 3, 5, 2, 4, 6).reshape(B, N // 64, 64)
    order = torch.rand(B, N // 64, 64, device=DEVICE, generator=g) + split(last)
    share = case['done'] * split(~last).sum(-1) + torch.rand(B, N // 64, device=DEVICE, generator=g)
    done = order.argsort(-1).argsort(-1) < share.floor()[..., None]
    done = done.view(B, shape[0] // 4, 4, 4, 4, 4, 4).permute(0, 1, 4, 2, 5, 3, 6).reshape(B, N)
    tokens = torch.where(done, torch.randint(C, (B, N), device=DEVICE, generator=g), torch.full((), C, device=DEVICE))
    orders = [torch.randperm(N // 64, device=DEVICE, generator=g) for _ in range(B)]
    return logits, tokens, last, done, orders


def _step_inputs(case, seed):
    g = _generator(seed)
    model = synth.StepModel(seed=seed % 1000)
    for p in model.parameters():
        p.data = p.data.to(torch.bfloat16)
    model = model.to(DEVICE)
    heads, width = model.cross[0].heads, model.cross[0].width
    conditions = []
    for L in _lengths(case):
        local = L - 4096
        prefix = [(_normal(g, heads, 4096, width // heads), _normal(g, heads, 4096, width // heads))
                  for _ in model.cross]
        positions = torch.rand(1, local, 3, device=DEVICE, generator=g) * torch.tensor([16., 64., 16.], device=DEVICE)
        conditions.append(Encoded(prefix, torch.randn(1, local, width, device=DEVICE, generator=g), positions))
    return model, conditions, _world(g, (case['windows'], 256, 16, 16), 304, 0.5)


# ------------------------------------------------------------------------------------------------ the measured calls

def prepare(case, seed):
    kind = case['kind']
    if kind == 'attend':
        query, windows = _attend_inputs(case, seed)
        context = CachedContext(1, case['windows'], case['heads'], case['head_dim'], max(_lengths(case)), DEVICE,
                                case['cache'])
        for b, (key, value) in enumerate(windows):
            context.write(0, b, key, value)
        return dict(kind=kind, context=context, query=query.transpose(1, 2), out=torch.empty_like(query).transpose(1, 2))
    if kind == 'masked':
        query, key, value, mask = _masked_inputs(case, seed)
        return dict(kind=kind, query=query, key=key, value=value, mask=mask)
    if kind == 'write':
        kv, positions, prefix = _write_inputs(case, seed)
        context = CachedContext(1, 1, case['heads'], case['head_dim'], case['capacity'], DEVICE, case['cache'])
        return dict(kind=kind, context=context, key=kv[:, 0].transpose(0, 1), value=kv[:, 1].transpose(0, 1),
                    prefix=prefix, positions=positions, frequencies=_frequencies(case['head_dim']))
    if kind == 'block':
        block, x, time, positions = _block_inputs(case, seed)
        return dict(kind=kind, block=block, x=x, time=time, positions=positions)
    if kind == 'patchify':
        conv, tokens = _patchify_inputs(case, seed)
        return dict(kind=kind, patch=GatherPatch(conv), tokens=tokens)
    if kind == 'select':
        logits, tokens, last, done, orders = _select_inputs(case, seed)
        B, N, C = logits.shape
        shape = (case['height'], 16, 16)
        select = EaseSelect(B, shape, C, 4, DEVICE)
        select.tokens.copy_(tokens)
        committed, free = done.sum(1).tolist(), (~last).sum(1).tolist()
        for b in range(B):
            select.bind_window(b, orders[b], last[b])
            k = min(N // 25, free[b] - committed[b])
            select.set_step(b, k, committed[b], (committed[b] + k) / free[b])
        if case['layout'] == 'patch':
            logits = PatchLogits(logits.view(B, N // 64, 64 * C), shape, 4, C)
        elif case['layout'] == 'planes':
            logits = logits.transpose(1, 2).contiguous().view(B, C, *shape)
        return dict(kind=kind, select=select, logits=logits)
    model, conditions, tokens = _step_inputs(case, seed)
    engine = SlotEngine(model, synth.WindowSpec(), DEVICE, case['windows'], l1_cap=8, l2_cap=256)
    for b, condition in enumerate(conditions):
        engine.load_slot(b, condition)
    engine.wait_loads()
    engine.tokens.copy_(tokens)
    return dict(kind=kind, engine=engine)


def run(state):
    kind = state['kind']
    if kind == 'attend':
        return state['context'].attend(0, state['query'], out=state['out'])
    if kind == 'masked':
        return attention(state['query'], state['key'], state['value'], key_mask=state['mask'])
    if kind == 'write':
        context = state['context']
        context.write(0, 0, state['key'], state['value'], prefix=state['prefix'], positions=state['positions'],
                      frequencies=state['frequencies'])
        if context.kv_dtype == 'bf16':
            return context.k[0], context.vt[0], context.lengths
        return (context.k[0].view(torch.uint8), context.vt[0].view(torch.uint8), context.k_scale[0],
                context.v_scale[0], context.lengths)
    if kind == 'block':
        with torch.inference_mode():
            return run_block(state['block'], state['x'], state['time'], state['positions'])
    if kind == 'patchify':
        return state['patch'](state['tokens'])
    if kind == 'select':
        select = state['select']
        select.run(state['logits'], keep_scores=True)
        return select.chosen, select.bad, select.scores
    return state['engine'].replay(0.5).patches


# --------------------------------------------------------------------------------------------------- what it takes

def work(case):
    kind = case['kind']
    if kind == 'attend':
        H, D, B, Q, keys = case['heads'], case['head_dim'], case['windows'], case['queries'], sum(_lengths(case))
        wide = 1 if case['cache'] == 'fp8' else 2
        return dict(bytes=2 * 2 * B * H * Q * D + 2 * wide * H * D * keys, flops=4 * H * D * Q * keys)
    if kind == 'masked':
        H, D, B, Q = case['heads'], case['head_dim'], case['windows'], case['queries']
        keys = sum(p + l for p, l in _valid(case))
        wide = 4 if case['dtype'] == 'fp32' else 2
        return dict(bytes=2 * wide * H * D * (B * Q + keys) + B * (case['prefix'] + case['local']),
                    flops=4 * H * D * Q * keys)
    if kind == 'write':
        H, D, keys = case['heads'], case['head_dim'], case['prefix'] + case['local']
        capacity = case['capacity'] + (-case['capacity']) % 64
        wide = 1 if case['cache'] == 'fp8' else 2
        return dict(bytes=2 * H * D * (2 * keys + wide * capacity) + 12 * case['local'],
                    flops=3 * H * D * case['local'])
    if kind == 'block':
        rows, W, N = case['windows'] * case['tokens'], case['width'], case['tokens']
        return dict(bytes=2 * (2 * rows * W + (12 + 6 * case['timed']) * W * W),
                    flops=24 * rows * W * W + 4 * rows * N * W + 12 * case['timed'] * case['windows'] * W * W)
    if kind == 'patchify':
        voxels, W = case['windows'] * case['height'] * 256, case['width']
        return dict(bytes=8 * voxels + 2 * W * ((case['classes'] + 1) * 64 + voxels // 64), flops=voxels * W)
    if kind == 'select':
        voxels, C = case['windows'] * case['height'] * 256, case['classes']
        wide = 4 if case['dtype'] == 'fp32' else 2
        return dict(bytes=voxels * (C * wide + 8 + 1 + 1 + 4), flops=5 * voxels * C)
    rows, keys = 1024 * case['windows'], sum(_lengths(case))
    blocks = 25 * 12 * 768 ** 2 + 13 * (12 + 2) * 384 ** 2 + 13 * 384 * 768 + 768 * 64 * 304
    cache = 13 * 2 * 384 * keys
    return dict(bytes=2 * (blocks + cache + 64 * 305 * (768 + 384) + 64 * 304 * rows + 6 * 25 * 768 ** 2),
                flops=2 * rows * blocks + 4 * rows * 1024 * (25 * 768 + 13 * 384) + 2 * 1024 * cache)


def tolerance(case):
    kind = case['kind']
    if kind in ('attend', 'masked'):
        # One rounding of P and one of the result to bf16 (2.3e-3 from the exact result); fp32 throughout otherwise
        # (7e-7 at 9744 keys, in another order of the sums a few times that).
        return dict(rel=1e-5) if case.get('dtype') == 'fp32' else dict(rel=1e-2)
    if kind == 'write':
        return 'exact'
    if kind in ('block', 'patchify'):
        return dict(rel=1e-2)            # 2.5e-3 and 2.3e-3 from the exact results
    if kind == 'select':
        # Voxels whose scores differ by a rounding may change places at a block's quota.
        return dict(rel=1e-6, differ=1e-4)
    return dict(rel=4e-2)                # 38 blocks of bf16 roundings: 1.2e-2 from the exact logits


# ------------------------------------------------------------------------------------------------------ in 64 bits

def _softmax_attention(q, k, v, keep=None):
    """q [H, Q, D], k and v [H, L, D] -> [H, Q, D] in float64."""
    scores = q.double() @ k.double().transpose(1, 2) / math.sqrt(q.shape[-1])
    if keep is not None:
        scores = scores.masked_fill(~keep, -math.inf)
    return scores.softmax(-1) @ v.double()


def _rotate(x, positions, frequencies):
    """AxialRoPE of x [..., N, D] at positions [N, 3], float64."""
    D = x.shape[-1]
    phase = (positions.double()[:, :, None] * frequencies.double()).reshape(-1, D // 2)
    even, odd, cos, sin = x[..., ::2], x[..., 1::2], phase.cos(), phase.sin()
    return torch.stack((even * cos - odd * sin, even * sin + odd * cos), -1).flatten(-2)


def _linear(layer, x):
    return torch.nn.functional.linear(x, layer.weight.double(), layer.bias.double())


def _norm(x, norm):
    weight, bias = (None if p is None else p.double() for p in (norm.weight, norm.bias))
    return torch.nn.functional.layer_norm(x, x.shape[-1:], weight, bias, norm.eps)


def _mlp(layers, x):
    return _linear(layers[2], torch.nn.functional.gelu(_linear(layers[0], x)))


def _block(block, x, time, positions):
    """One window: x [N, W], time [W] or None, positions [N, 3]."""
    N, W = x.shape
    H = block.attn.heads
    if time is None:
        one = torch.ones((), dtype=torch.float64, device=x.device)
        s1 = c1 = s2 = c2 = 0 * one
        g1 = g2 = one
    else:
        s1, c1, g1, s2, c2, g2 = _linear(block.ada[1], torch.nn.functional.silu(time)).chunk(6, -1)
    q, k, v = _linear(block.attn.qkv, _norm(x, block.norm1) * (1 + c1) + s1).view(N, 3, H, W // H).permute(1, 2, 0, 3)
    q, k = (_rotate(t, positions, block.attn.rope.frequencies) for t in (q, k))
    x = x + g1 * _linear(block.attn.proj, _softmax_attention(q, k, v).transpose(0, 1).reshape(N, W))
    return x + g2 * _mlp(block.mlp, _norm(x, block.norm2) * (1 + c2) + s2)


def _embed(conv, tokens):
    """tokens [Y, Z, X] -> [patches, W]: the weight rows that the voxels pick, summed, as the bf16 tables hold them."""
    Y, Z, X = tokens.shape
    table = conv.weight.detach().to(torch.bfloat16).permute(1, 2, 3, 4, 0).flatten(1, 3).double()
    voxels = tokens.view(Y // 4, 4, Z // 4, 4, X // 4, 4).permute(0, 2, 4, 1, 3, 5).reshape(-1, 64)
    out = sum(table[:, o][voxels[:, o]] for o in range(64))
    return out + conv.bias.detach().to(torch.bfloat16).double()


def _e4m3(x):
    """Codes and scale of one window's x [H, L, D], a scale for each head."""
    scale = torch.clamp(x.float().abs().amax((1, 2)) / 448.0, min=1e-12)
    return (x.float() / scale[:, None, None]).to(torch.float8_e4m3fn), scale


def _step(model, condition, tokens):
    """One window of the streaming ControlNet's forward at timestep 0.5."""
    bb, cc = model.backbone, model.control
    prefix, local, local_positions = condition
    origin = torch.tensor([0.0, -64.0, 0.0], device=DEVICE)
    centers = bb.patch_centers_xyz + origin
    own, shared = bb.patch_centers_xyz / 4, (centers - origin) / 4
    y = (2 * (centers[:, 1:2] - bb.y_range[0]) / (bb.y_range[1] - bb.y_range[0]) - 1).double()

    def start(trunk):
        t = torch.tensor([0.5], device=DEVICE)
        half = trunk.time_dim // 8
        phase = t.double()[:, None] * torch.exp(-math.log(10000.0) * torch.arange(half, device=DEVICE).double() / half)
        time = _mlp(trunk.time_mlp, torch.cat((phase.sin(), phase.cos()), -1))
        time = _linear(trunk.time_projection[1], torch.nn.functional.silu(time))[0]
        rise = _linear(trunk.y_embed[2], torch.nn.functional.silu(_linear(trunk.y_embed[0], y)))
        return _embed(trunk.target_patch, tokens) + rise, time

    (b, bt), (c, ct) = start(bb), start(cc)
    for i in range(bb.depth):
        b = _block(bb.blocks[i], b, bt, own)
        j = model.layer_map.get(i)
        if j is None:
            continue
        c = _block(cc.blocks[j], c, ct, own)
        cross = model.cross[j]
        N, W = c.shape
        split = lambda x: x.view(len(x), cross.heads, -1).transpose(0, 1)
        q = _rotate(split(_linear(cross.query, _norm(c, cross.norm))), shared, cross.rope.frequencies)
        key, value = _linear(cross.key_value, local[0].to(torch.bfloat16).double()).chunk(2, -1)
        key = _rotate(split(key), local_positions[0], cross.rope.frequencies)
        key, value = torch.cat((prefix[j][0].double(), key), 1), torch.cat((prefix[j][1].double(), split(value)), 1)
        c = c + _linear(cross.proj, _softmax_attention(q, key, value).transpose(0, 1).reshape(N, W))
        b = b + _linear(model.zero[j], c)
    shift, gain = _linear(bb.final_ada[1], torch.nn.functional.silu(bt)).chunk(2, -1)
    return _linear(bb.class_head, _norm(b, bb.final_norm) * (1 + gain) + shift)


@torch.inference_mode()
def exact(case, seed):
    kind = case['kind']
    if kind == 'attend':
        query, windows = _attend_inputs(case, seed)
        out = torch.empty(case['windows'], case['heads'], case['queries'], case['head_dim'], dtype=torch.float64,
                          device=DEVICE)
        for b, (key, value) in enumerate(windows):
            if case['cache'] == 'fp8':
                key, value = (codes.double() * scale.double()[:, None, None]
                              for codes, scale in (_e4m3(key), _e4m3(value)))
            out[b] = _softmax_attention(query[b].transpose(0, 1), key, value)
        return out
    if kind == 'masked':
        query, key, value, mask = _masked_inputs(case, seed)
        return torch.stack([_softmax_attention(*window) for window in zip(query, key, value, mask)])
    if kind == 'write':
        return None                      # copies and codes: compared bit for bit
    if kind == 'block':
        block, x, time, positions = _block_inputs(case, seed)
        return torch.stack([_block(block, x[b].double(), None if time is None else time[b].double(), positions[b])
                            for b in range(len(x))])
    if kind == 'patchify':
        conv, tokens = _patchify_inputs(case, seed)
        return torch.stack([_embed(conv, t) for t in tokens])
    if kind == 'select':
        logits = _select_inputs(case, seed)[0]
        scores = torch.stack([-torch.special.entr(x.double().softmax(-1)).sum(-1) for x in logits])
        if case['layout'] == 'patch':
            # Row r of the class head is voxel r of patch order; the scores lie in (y, z, x) order.
            B, Y = case['windows'], case['height']
            scores = scores.view(B, Y // 4, 4, 4, 4, 4, 4).permute(0, 1, 4, 2, 5, 3, 6).reshape(B, -1)
        return None, None, scores
    model, conditions, tokens = _step_inputs(case, seed)
    return torch.stack([_step(model, condition, t) for condition, t in zip(conditions, tokens)])
