"""The key split of the cross attention against the float64 oracle and against the unsplit launch of the same call.

Window lengths where the split can go wrong: ranges that end on a unit's first and last block, one block past the
length from which windows are split, empty windows between long ones, a single window cut into many parts, parts that
a key mask empties. The bars are the unsplit kernels' (bf16 2e-2 and 1e-2 of the largest value, fp32 2e-5 and 1e-4: the
parts are kept and joined in fp32, so the split adds no rounding of its own to them)."""
import math

import pytest
import torch

from oracle import attention as A

pytestmark = pytest.mark.gpu

EDGE = 24 * 64                      # the keys from which a window is split


def _case(msg):
    print(f'[gpu-case] {msg}', flush=True)


@pytest.fixture(scope='module')
def dev():
    if not torch.cuda.is_available():
        pytest.skip('no GPU')
    import streamvoxel_amd
    streamvoxel_amd.load()
    return torch.device('cuda:0')


def qkv(B, H, Q, kcap, D, seed, dtype, spread=1.0):
    g = torch.Generator().manual_seed(seed)
    s = spread / math.sqrt(D)
    return [(torch.randn(B, H, n, D, generator=g) * s).to(dtype) for n in (Q, kcap, kcap)]


def check(got, ref, atol, rtol):
    err = (got.double().cpu() - ref).abs().max().item()
    assert err <= atol and err <= rtol * ref.abs().max().item(), (err, ref.abs().max().item())


LENGTHS = [[EDGE - 64, 1, 0, 700],                       # no window is split
           [EDGE - 63], [EDGE], [EDGE + 1],              # the edge itself
           [6000],                                       # one window, many parts
           [0, 5000, 0, 0, 1, 4097, 64, 0],              # empty and short windows between long ones
           [2048, 2048, 2048, 2048]]                     # equal ranges


@pytest.mark.parametrize('lengths', LENGTHS, ids=lambda x: '-'.join(map(str, x)))
@pytest.mark.parametrize('D,H,Q', [(48, 3, 130), (64, 4, 128), (96, 2, 257), (128, 1, 33)])
def test_split_windows_match_the_oracle(dev, lengths, D, H, Q):
    from streamvoxel_amd import _lib
    from streamvoxel_amd.stream.attention import attention
    _case(f'split bf16 D={D} H={H} Q={Q} lengths={lengths}')
    B, kcap = len(lengths), max(lengths) + 5
    kcap += -kcap % 8
    q, k, v = qkv(B, H, Q, kcap, D, sum(lengths) + D, torch.bfloat16, 2.0)
    assert int(_lib.load().svhip_xattn_workspace_bytes(B, H, Q, D, kcap)) > 0
    ref = A.cross_attention(q, k, v, lengths)
    lt = torch.tensor(lengths, dtype=torch.int32, device=dev)
    qd, kd, vd = q.to(dev), k.to(dev), v.to(dev)
    out = attention(qd, kd, vd, lengths=lt)
    out_t = attention(qd, kd, vd.transpose(2, 3).contiguous().transpose(2, 3), lengths=lt)
    mask = torch.arange(kcap, device=dev)[None] < lt[:, None]
    out_m = attention(qd, kd, vd, key_mask=mask)
    cu = torch.tensor([0] + torch.tensor(lengths).cumsum(0).tolist(), dtype=torch.int32, device=dev)
    kp, vp = (torch.cat([x[b, :, :n] for b, n in enumerate(lengths)], 1).contiguous() for x in (kd, vd))
    out_p = attention(qd, kp, vp, cu_seqlens=cu)
    torch.cuda.synchronize()
    check(out, ref, 2e-2, 1e-2)
    for b, n in enumerate(lengths):
        if n == 0:
            assert not out[b].any()
    # Every layout of the same keys is cut alike and gives the same bits.
    assert torch.equal(out, out_t) and torch.equal(out, out_m) and torch.equal(out, out_p)


@pytest.mark.parametrize('D', [48, 64])
def test_split_under_masks_with_holes(dev, D):
    from streamvoxel_amd.stream.attention import attention
    B, H, Q, kcap = 4, 3, 140, 4000
    _case(f'split bf16 key mask D={D}')
    q, k, v = qkv(B, H, Q, kcap, D, D, torch.bfloat16, 2.0)
    g = torch.Generator().manual_seed(D)
    mask = torch.rand(B, kcap, generator=g) < 0.5
    mask[0, 200:3000] = False                     # whole parts of the window masked
    mask[1] = False                               # no attended key at all
    mask[2, :3900] = False                        # only the last part holds attended keys
    scores = (q.double() @ k.double().transpose(2, 3)) / math.sqrt(D)
    w = scores.masked_fill(~mask[:, None, None], -math.inf).softmax(-1).nan_to_num(0.0)
    ref = w @ v.double()
    out = attention(q.to(dev), k.to(dev), v.to(dev), key_mask=mask.to(dev))
    torch.cuda.synchronize()
    assert not out[1].any()
    check(out, ref, 2e-2, 1e-2)


@pytest.mark.parametrize('vt', [False, True])
def test_e4m3_is_not_split(dev, vt):
    """A window over an e4m3 cache gives the same bits alone and in a batch, also where its sizes would be split."""
    from streamvoxel_amd.stream.attention import attention, quantize_e4m3
    lengths = [4000, 0, 2500, 63]
    B, H, Q, D, kcap = 4, 4, 200, 64, 4032
    _case(f'e4m3 alone and in a batch vt={vt}')
    q, k, v = (x.to(dev) for x in qkv(B, H, Q, kcap, D, 3, torch.bfloat16, 2.0))
    (kc, ks), (vc, vs) = quantize_e4m3(k), quantize_e4m3(v)
    if vt:
        vc = vc.transpose(2, 3).contiguous().transpose(2, 3)
    lt = torch.tensor(lengths, dtype=torch.int32, device=dev)
    out = attention(q, kc, vc, lengths=lt, k_scale=ks, v_scale=vs)
    for b in range(B):
        one = attention(q[b:b + 1], kc[b:b + 1], vc[b:b + 1], lengths=lt[b:b + 1], k_scale=ks[b:b + 1],
                        v_scale=vs[b:b + 1])
        torch.cuda.synchronize()
        assert torch.equal(one, out[b:b + 1])


def check_alone_and_in_batches(dev, q, k, v, lengths, batches):
    """Every window of `lengths` attended alone and in each of `batches` (lists of window indices): the same bits, as
    rows of padded K/V and under the key mask of the same lengths."""
    from streamvoxel_amd.stream.attention import attention
    lt = torch.tensor(lengths, dtype=torch.int32, device=dev)
    mask = torch.arange(k.shape[2], device=dev)[None] < lt[:, None]
    alone = [attention(q[b:b + 1], k[b:b + 1], v[b:b + 1], lengths=lt[b:b + 1]) for b in range(len(lengths))]
    for at in [[b] for b in range(len(lengths))] + batches:
        out = attention(q[at], k[at], v[at], lengths=lt[at])
        out_m = attention(q[at], k[at], v[at], key_mask=mask[at])
        torch.cuda.synchronize()
        for i, b in enumerate(at):
            assert torch.equal(out[i:i + 1], alone[b]), (at, b)
            assert torch.equal(out_m[i:i + 1], alone[b]), ('mask', at, b)


# Lengths short of the first cut, on it, at and past the piece counts that follow, with and without a partial block.
ALONE = [EDGE - 64, EDGE - 63, EDGE + 130, 0, 30 * 64, 4097, 6400, 63]
# Batches: some, with repetitions that fill the chip (unsplit) or go past one wave's windows (unsplit).
BATCHES = [[0, 1], [2, 4, 6], list(range(8)), list(range(8)) * 6, list(range(8)) * 9]


@pytest.mark.parametrize('D,H,Q', [(48, 8, 1000), (64, 6, 1024), (96, 4, 700), (128, 2, 130), (64, 1, 20), (48, 2, 3300)])
@pytest.mark.parametrize('vt', [False, True])
def test_bf16_windows_alone_and_in_batches(dev, D, H, Q, vt):
    """Where a window is cut depends on itself alone: the same bits alone, in split batches of several sizes and in
    batches that are not split, over either V layout (head counts and query tiles for 16, 12, 8 pieces and none)."""
    _case(f'bf16 alone and in batches D={D} H={H} Q={Q} vt={vt}')
    q, k, v = (x.to(dev) for x in qkv(8, H, Q, 6400, D, D + H, torch.bfloat16, 2.0))
    if vt:
        v = v.transpose(2, 3).contiguous().transpose(2, 3)
    check_alone_and_in_batches(dev, q, k, v, ALONE, BATCHES[:4] if Q > 2000 else BATCHES)


@pytest.mark.parametrize('D,H,Q', [(16, 3, 130), (48, 8, 500), (64, 12, 1024)])
def test_fp32_windows_alone_and_in_batches(dev, D, H, Q):
    _case(f'fp32 alone and in batches D={D} H={H} Q={Q}')
    q, k, v = (x.to(dev) for x in qkv(8, H, Q, 6400, D, D + H, torch.float32, 2.0))
    check_alone_and_in_batches(dev, q, k, v, ALONE, BATCHES)


@pytest.mark.parametrize('dtype', ['bf16', 'fp32'])
def test_windows_under_masks_with_holes_alone_and_in_batches(dev, dtype):
    """The same under masks that leave out whole pieces, the window's end and every second block."""
    from streamvoxel_amd.stream.attention import attention
    H, Q, D, kcap = 6, 512, 64, 6000
    _case(f'masks alone and in batches {dtype}')
    q, k, v = (x.to(dev) for x in qkv(6, H, Q, kcap, D, 7, torch.bfloat16 if dtype == 'bf16' else torch.float32, 2.0))
    mask = torch.rand(6, kcap, generator=torch.Generator().manual_seed(4)) < 0.5
    mask[0, 200:4000] = False
    mask[1] = False
    mask[2, :5900] = False
    mask[3, 2500:] = False
    mask[4] = (torch.arange(kcap) // 64) % 2 == 1
    mask = mask.to(dev)
    alone = [attention(q[b:b + 1], k[b:b + 1], v[b:b + 1], key_mask=mask[b:b + 1]) for b in range(6)]
    for at in ([0, 4], list(range(6)), list(range(6)) * 4, list(range(6)) * 12):
        out = attention(q[at], k[at], v[at], key_mask=mask[at])
        torch.cuda.synchronize()
        for i, b in enumerate(at):
            assert torch.equal(out[i:i + 1], alone[b]), (at, b)


@pytest.mark.parametrize('lengths', LENGTHS, ids=lambda x: '-'.join(map(str, x)))
@pytest.mark.parametrize('D', [16, 32, 48, 64])
def test_split_fp32_windows_match_the_oracle(dev, lengths, D):
    from streamvoxel_amd.stream.attention import attention
    B, H, Q, kcap = len(lengths), 2, 130, max(lengths) + 4
    kcap += -kcap % 4
    _case(f'split fp32 D={D} lengths={lengths}')
    q, k, v = qkv(B, H, Q, kcap, D, sum(lengths) + D, torch.float32)
    ref = A.cross_attention(q, k, v, lengths)
    lt = torch.tensor(lengths, dtype=torch.int32, device=dev)
    qd, kd, vd = q.to(dev), k.to(dev), v.to(dev)
    out = attention(qd, kd, vd, lengths=lt)
    out_t = attention(qd, kd, vd.transpose(2, 3).contiguous().transpose(2, 3), lengths=lt)
    out_m = attention(qd, kd, vd, key_mask=torch.arange(kcap, device=dev)[None] < lt[:, None])
    torch.cuda.synchronize()
    check(out, ref, 2e-5, 1e-4)
    # Every layout of the same keys is cut alike and gives the same bits.
    assert torch.equal(out, out_t) and torch.equal(out, out_m)


def test_split_replays_in_a_graph(dev):
    """Captured: the scratch comes from the graph's pool, and lengths changed between replays are planned anew."""
    from streamvoxel_amd.stream.attention import attention
    B, H, Q, D, kcap = 2, 4, 128, 64, 6016
    _case('split in a graph')
    q, k, v = (x.to(dev) for x in qkv(B, H, Q, kcap, D, 9, torch.bfloat16, 2.0))
    lt = torch.tensor([6000, 100], dtype=torch.int32, device=dev)
    out = torch.empty_like(q)
    attention(q, k, v, lengths=lt, out=out)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        attention(q, k, v, lengths=lt, out=out)
    for lengths in ([6000, 100], [0, 6016], [64, 1500], [3000, 3001]):
        lt.copy_(torch.tensor(lengths, dtype=torch.int32))
        graph.replay()
        want = attention(q, k, v, lengths=lt)
        torch.cuda.synchronize()
        assert torch.equal(out, want), lengths


@pytest.mark.parametrize('cap', [1, 63, 64, 65, 1000, 70001])
def test_mask_blocks_against_torch(dev, cap):
    """Lengths and lists of attended blocks: capacities around a block and past one round of 1024 blocks, rows of any
    alignment, windows cut by kv_len, empty ones."""
    from streamvoxel_amd import _lib
    g = torch.Generator().manual_seed(cap)
    B, nb = 5, (cap + 63) // 64
    mask = torch.rand(B, cap + 3, generator=g) < 0.02
    mask[1] = True
    mask[2] = False
    lens = torch.tensor([cap, cap, cap, cap // 2, 0], dtype=torch.int32)
    dm = mask.to(dev)
    lib = _lib.load()
    for given in (False, True):
        _case(f'mask blocks cap={cap} lengths={given}')
        out = torch.full((B,), -7, dtype=torch.int32, device=dev)
        blocks = torch.full((B, nb + 2), -7, dtype=torch.int32, device=dev)
        dl = lens.to(dev)
        _lib.check(lib.svhip_mask_blocks(_lib.ptr(dm.view(torch.uint8)), dm.stride(0), _lib.ptr(dl) if given else None, B,
                                         cap, _lib.ptr(out), _lib.ptr(blocks), nb + 2, _lib.stream_of(dm)),
                   'svhip_mask_blocks')
        torch.cuda.synchronize()
        for b in range(B):
            row = mask[b, :int(lens[b]) if given else cap]
            at = row.nonzero().flatten()
            want = sorted({int(i) // 64 for i in at})
            assert int(out[b]) == (int(at[-1]) + 1 if len(at) else 0)
            assert blocks[b, 0] == len(want) and blocks[b, 1:1 + len(want)].tolist() == want
            assert (blocks[b, 1 + len(want):] == -7).all()


@pytest.mark.parametrize('L', [40, 5000])
def test_fp32_rows_of_infinite_scores(dev, L):
    """A query whose every score is -inf, or that meets +inf, gets NaN without a key mask, as torch's softmax gives;
    the other queries of its tile are untouched (unsplit and split lengths)."""
    from streamvoxel_amd.stream.attention import attention
    B, H, Q, D = 1, 2, 70, 64
    _case(f'fp32 infinite scores L={L}')
    q, k, v = qkv(B, H, Q, L, D, L, torch.float32)
    k[..., 0] = k[..., 0].abs() + 0.1
    clean = q.clone()
    q[0, 0, 3, 0], q[0, 1, 69, 0] = -math.inf, math.inf
    lt = torch.tensor([L], dtype=torch.int32, device=dev)
    out = attention(q.to(dev), k.to(dev), v.to(dev), lengths=lt).cpu()
    want = attention(clean.to(dev), k.to(dev), v.to(dev), lengths=lt).cpu()
    bad = torch.zeros(B, H, Q, dtype=torch.bool)
    bad[0, 0, 3] = bad[0, 1, 69] = True
    assert out[bad].isnan().all()
    # An infinite score may raise the running max of the wave it is in, never another query's.
    assert torch.allclose(out[~bad], want[~bad], rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize('D', [48, 64, 96])
@pytest.mark.parametrize('lengths', [[700], [6000], [5000, 40, 4000, 1600]], ids=lambda x: '-'.join(map(str, x)))
def test_nan_queries_stay_nan(dev, D, lengths):
    """A NaN query gives NaN rows, whether its window is attended whole or in parts; the queries of other waves (32
    queries each) keep their bits, the ones of the same wave may see their running max raised (the tile's bars). At
    head_dim 96 the row sums of queries c and c + 16 of a wave share an operand column, so query 21 is left out."""
    from streamvoxel_amd.stream.attention import attention
    B, H, Q, kcap = len(lengths), 2, 200, max(lengths) + 8
    _case(f'NaN queries D={D} lengths={lengths}')
    q, k, v = qkv(B, H, Q, kcap, D, D + B, torch.bfloat16)
    bad = torch.zeros(B, H, Q, dtype=torch.bool)
    bad[0, 1, 5] = bad[B - 1, 0, 199] = True
    qn = q.clone()
    qn[0, 1, 5] = math.nan
    qn[B - 1, 0, 199, 3] = math.nan
    lt = torch.tensor(lengths, dtype=torch.int32, device=dev)
    kd, vd = k.to(dev), v.to(dev)
    vt = vd.transpose(2, 3).contiguous().transpose(2, 3)
    same_wave = torch.zeros_like(bad)
    same_wave[0, 1, :32] = same_wave[B - 1, 0, 192:] = True
    for val in (vd, vt):
        want = attention(q.to(dev), kd, val, lengths=lt).cpu()
        got = attention(qn.to(dev), kd, val, lengths=lt).cpu()
        assert got[bad].isnan().all()
        assert torch.equal(got[~same_wave], want[~same_wave])
        near = same_wave & ~bad
        near[0, 1, 21] = False
        assert (got[near].float() - want[near].float()).abs().max() <= 2e-2


@pytest.mark.parametrize('workspace', [False, True])
def test_packed_lengths_win_over_kv_len(dev, workspace):
    """svhip_xattn_fwd and _ws given both kv_len and cu_seqlens: the packed lengths hold, kv_len is not read."""
    from streamvoxel_amd import _lib
    from streamvoxel_amd.stream.attention import attention
    lengths, H, Q, D = [2000, 500], 2, 130, 64
    _case(f'packed with kv_len workspace={workspace}')
    total = sum(lengths)
    q, k, v = (x.to(dev) for x in qkv(2, H, Q, total, D, 5, torch.bfloat16))
    kp, vp = k[0].contiguous(), v[0].contiguous()
    cu = torch.tensor([0, lengths[0], total], dtype=torch.int32, device=dev)
    lib = _lib.load()
    nbytes = int(lib.svhip_xattn_workspace_bytes(2, H, Q, D, total))
    assert nbytes > 0
    ws = torch.empty(nbytes, dtype=torch.uint8, device=dev) if workspace else None
    outs = []
    for kv_len in (None, torch.tensor([100, 7], dtype=torch.int32, device=dev)):
        out = torch.zeros_like(q)
        args = [_lib.ptr(q), _lib.ptr(kp), _lib.ptr(vp), _lib.ptr(out), _lib.SVHIP_BF16, _lib.ptr(kv_len), _lib.ptr(cu),
                None, None, 2, H, Q, D, total, *q.stride()[:3], 0, *kp.stride()[:2], 0, *vp.stride(), *out.stride()[:3],
                1.0 / math.sqrt(D)]
        if workspace:
            rc = lib.svhip_xattn_fwd_ws(*args, _lib.ptr(ws), nbytes, _lib.stream_of(q))
        else:
            rc = lib.svhip_xattn_fwd(*args, _lib.stream_of(q))
        _lib.check(rc, 'svhip_xattn_fwd')
        torch.cuda.synchronize()
        outs.append(out)
    assert torch.equal(outs[0], outs[1])
    if workspace:
        assert torch.equal(outs[0], attention(q, kp, vp, cu_seqlens=cu))


@pytest.mark.parametrize('lengths', [False, True])
def test_fp32_fully_masked_window_with_a_list(dev, lengths):
    """One fp32 window without an attended key, its list of blocks given with and without its length: zeros, whatever
    the scratch holds (zeros where an entry could be taken for a team or a slot, ones elsewhere)."""
    from streamvoxel_amd import _lib
    H, Q, D, kcap = 2, 130, 64, 4000
    _case(f'fp32 empty list lengths={lengths}')
    q, k, v = (x.to(dev) for x in qkv(1, H, Q, kcap, D, 1, torch.float32))
    mask = torch.zeros(1, kcap, dtype=torch.uint8, device=dev)
    cut = torch.zeros(1, dtype=torch.int32, device=dev)
    blocks = torch.zeros(1, 1 + (kcap + 63) // 64, dtype=torch.int32, device=dev)
    lib = _lib.load()
    nbytes = int(lib.svhip_xattn_f32_workspace_bytes(1, H, Q, D, kcap))
    assert nbytes > 0
    ws = torch.ones(nbytes // 4, dtype=torch.float32, device=dev)
    ws[-2 * H:] = 0
    out = torch.full_like(q, 7.0)
    _lib.check(lib.svhip_xattn_fwd_f32_ws(
        _lib.ptr(q), _lib.ptr(k), _lib.ptr(v), _lib.ptr(out), _lib.ptr(mask), kcap, _lib.ptr(cut) if lengths else None,
        _lib.ptr(blocks), blocks.stride(0), None, 1, H, Q, D, kcap, *q.stride()[:3], *k.stride()[:3], *v.stride(),
        *out.stride()[:3], 0.125, _lib.ptr(ws), nbytes, _lib.stream_of(q)), 'svhip_xattn_fwd_f32_ws')
    torch.cuda.synchronize()
    assert not out.any()


@pytest.mark.parametrize('dtype,D', [('bf16', 48), ('bf16', 64), ('bf16', 96), ('bf16', 128), ('fp32', 48), ('fp32', 64)])
@pytest.mark.parametrize('lengths', [[6000], [6000, 2000, 4096]], ids=lambda x: '-'.join(map(str, x)))
def test_stretch_of_minus_infinite_scores(dev, dtype, D, lengths):
    """Queries whose scores are -inf (by overflow of the score product) over most of the window, from its second block
    to its last but one: those keys weigh nothing, wherever the window is cut, and the rows stay finite."""
    from streamvoxel_amd.stream.attention import attention
    dt = torch.bfloat16 if dtype == 'bf16' else torch.float32
    B, H, Q, kcap = len(lengths), 2, 140, max(lengths)
    _case(f'-inf stretch {dtype} D={D} lengths={lengths}')
    q, k, v = qkv(B, H, Q, kcap, D, D, torch.float32)
    q[..., 0], k[..., 0] = 0.0, 0.0
    bad = torch.zeros(B, H, Q, dtype=torch.bool)
    bad[:, :, ::7] = True
    q[..., 0][bad] = 3e38
    for b, n in enumerate(lengths):
        k[b, :, 64:n - 100, 0] = -3e38
    q, k, v = (x.to(dt) for x in (q, k, v))
    ref = A.cross_attention(q, k, v, lengths)
    out = attention(q.to(dev), k.to(dev), v.to(dev), lengths=torch.tensor(lengths, dtype=torch.int32, device=dev))
    torch.cuda.synchronize()
    assert bool(out.isfinite().all())
    check(out, ref, *((2e-2, 1e-2) if dtype == 'bf16' else (2e-5, 1e-4)))
