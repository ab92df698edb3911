"""dtree_causal_attention (one launch per prompt segment) against float64.

Both head geometries, prefixes and segments that end inside a page, a 32-row
block and a workgroup's four (row block, head) pairs, group sizes 2 to 8, both
output layouts, permuted pages, and NaN in every cache slot the segment does
not own. Outputs are compared as hi + lo pairs: q and P carry 16 significant
bits, so a score of up to |q| |k| scale = 11 is off by 2^-16 * 11 and an output
by about that share of |v|: 2e-4 relative to the output's norm (measured 3e-5);
K and V rows are the bf16 rounding of the exact ones up to one flip."""
import ctypes as C

import pytest
import torch

from dtree_hip import _native as N
from dtree_hip.cache import PagedKVCache
from dtree_hip.weights import untile_weight

pytestmark = pytest.mark.gpu


def _rope(x, pos, dims, base):
    half = dims // 2
    inv = base ** (-torch.arange(half, dtype=torch.float64, device=x.device) * 2.0 / dims)
    ang = pos.double()[:, None] * inv
    c, s = torch.cos(ang)[:, None], torch.sin(ang)[:, None]
    a, b = x[..., :half], x[..., half:dims]
    return torch.cat([a * c - b * s, a * s + b * c, x[..., dims:]], -1)


def _case(dev, geo, Hq, Hkv, past, n, tiled=True, norms=True, workspace=None, pad=32, norm_off=0):
    """workspace: None, or (bytes, misalignment) for dtree_causal_attention_split;
    returns the share of the workspace that the call wrote. pad: rows of qkv and
    out come in multiples of it."""
    D, R, gated = (128, 128, 0) if geo == "qwen3" else (256, 64, 1)
    g = torch.Generator(device=dev)
    g.manual_seed(past * 1000 + n + Hq)
    rnd = lambda *s: torch.empty(*s, device=dev).normal_(generator=g)  # noqa: E731
    rows = pad * ((n + pad - 1) // pad)
    qs = D * (2 if gated else 1)
    ld = Hq * qs + 2 * Hkv * D
    qkv = torch.zeros(rows, ld, device=dev)
    qkv[:n] = rnd(n, ld)
    qn, kn = ((1 + 0.1 * rnd(D + norm_off)).to(torch.bfloat16)[norm_off:] for _ in range(2))
    npages = (past + n + 63) // 64 + 2
    cache = PagedKVCache(1, Hkv, D, 64 * npages, device=dev,
                         page_order=torch.randperm(npages, generator=torch.Generator().manual_seed(n)))
    cache.k_pages.fill_(float("nan"))
    cache.v_pages.fill_(float("nan"))
    kpre, vpre = (rnd(past, Hkv, D).to(torch.bfloat16) for _ in range(2))
    if past:
        cache.write_logical(0, kpre, vpre)
    cos, sin = (torch.zeros(rows, R // 2, device=dev) for _ in range(2))
    st = torch.cuda.current_stream().cuda_stream
    base = 1e5
    N.call("dtree_rope_positions", past, rows, R, base, cos.data_ptr(), sin.data_ptr(), st)
    width = Hq * D
    out = torch.full((2, rows, width), float("nan"), dtype=torch.bfloat16, device=dev)
    a = N.AttnArgs()
    a.qkv = qkv.data_ptr(); a.ld_qkv = ld
    if norms:
        a.q_norm, a.k_norm = qn.data_ptr(), kn.data_ptr()
    a.eps = 1e-6
    a.rope_cos, a.rope_sin = cos.data_ptr(), sin.data_ptr()
    a.k_pages, a.v_pages, a.page_table = cache.k_ptr(0), cache.v_ptr(0), cache.page_table.data_ptr()
    a.out, a.out_lo = out[0].data_ptr(), out[1].data_ptr()
    a.ld_out = width; a.out_layout = N.W_TILED if tiled else N.W_ROWMAJOR
    a.num_heads, a.num_kv_heads, a.head_dim, a.rows_padded = Hq, Hkv, D, rows
    a.scale = D ** -0.5; a.rope_dims = R; a.gated = gated
    print(f"causal attention {geo} Hq={Hq} Hkv={Hkv} past={past} n={n} tiled={tiled} {workspace}", flush=True)
    if workspace is None:
        N.check(N.lib().dtree_causal_attention(C.byref(a), past, n, st), "causal attention")
    else:
        ws = torch.full((workspace[0] // 4 + 4,), float("nan"), device=dev)
        N.check(N.lib().dtree_causal_attention_split(C.byref(a), past, n, ws.data_ptr() + workspace[1], workspace[0],
                                                     st), "causal attention")
    torch.cuda.synchronize()

    x = qkv[:n].double()
    rms = lambda t, w: t * torch.rsqrt(t.square().mean(-1, keepdim=True) + 1e-6) * w.double()  # noqa: E731
    q = x[:, :Hq * qs].reshape(n, Hq, qs)
    gate, q = q[..., D:], q[..., :D]
    k = x[:, Hq * qs:Hq * qs + Hkv * D].reshape(n, Hkv, D)
    v = x[:, Hq * qs + Hkv * D:].reshape(n, Hkv, D)
    if norms:
        q, k = rms(q, qn), rms(k, kn)
    pos = torch.arange(past, past + n, device=dev)
    q, k = _rope(q, pos, R, base), _rope(k, pos, R, base)
    got_k, got_v = cache.logical_keys(0, past + n), cache.logical_values(0, past + n)
    assert torch.equal(got_k[:past], kpre) and torch.equal(got_v[:past], vpre)
    assert ((got_k[past:].double() - k).abs() <= 2.0 ** -8 * k.abs() + 1e-6).all()
    assert torch.equal(got_v[past:], qkv[:n, Hq * qs + Hkv * D:].reshape(n, Hkv, D).to(torch.bfloat16))
    # slots past the segment are untouched
    rest = cache.logical_keys(0, 64 * npages)[past + n:], cache.logical_values(0, 64 * npages)[past + n:]
    assert all(torch.isnan(t).all() for t in rest)
    K, V = got_k.double(), got_v.double()
    s = torch.einsum("nhd,khd->hnk", q, K.repeat_interleave(Hq // Hkv, 1)) * D ** -0.5
    vis = torch.arange(past + n, device=dev)[None] <= pos[:, None]
    w = torch.softmax(s.masked_fill(~vis[None], float("-inf")), -1)
    ref = torch.einsum("hnk,khd->nhd", w, V.repeat_interleave(Hq // Hkv, 1))
    if gated:
        ref = ref * torch.sigmoid(gate)
    o = out.double() if not tiled else torch.stack([untile_weight(t).double() for t in out])
    o = o[0] + o[1]
    assert (o[n:] == 0).all()
    err = ((o[:n] - ref.reshape(n, -1)).norm() / ref.norm()).item()
    assert err <= 2e-4, err
    if workspace is not None:
        assert torch.isnan(ws[workspace[0] // 4:]).all()
        used = 1 - torch.isnan(ws).double().mean().item()
        # captured, with eager work between the replays and stale buffers each time
        first, graph = out.clone(), torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            N.check(N.lib().dtree_causal_attention_split(C.byref(a), past, n, ws.data_ptr() + workspace[1], workspace[0],
                                                         torch.cuda.current_stream().cuda_stream), "causal attention")
        for _ in range(3):
            out.fill_(float("nan"))
            ws.fill_(float("nan"))
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, first)
        return used


# partial results of one key range: per workgroup (four 32-row units), O and two statistics
def _range_bytes(Hq, Hkv, D, n):
    return Hkv * ((Hq // Hkv * ((n + 31) // 32) + 3) // 4) * 4 * (32 * D + 64) * 4


@pytest.mark.parametrize("geo,D", [("qwen3", 128), ("gated", 256)])
@pytest.mark.parametrize("past,n", [(300, 1), (0, 200), (448, 64), (383, 66), (1000, 31), (4095, 33), (1985, 130),
                                    (127, 513)])
def test_causal_key_ranges(gpu_device, geo, D, past, n):
    """Prefixes that end inside a page, rows whose first keys lie past some
    ranges, empty last ranges; pages the segment does not own hold NaN."""
    full = N.lib().dtree_causal_attention_workspace_bytes(D)
    pages = (past + n + 63) // 64
    used = _case(gpu_device, geo, 8, 2, past, n, workspace=(full, 0))
    assert (used > 0) == (pages >= (8 if D == 128 else 4))


@pytest.mark.parametrize("geo,D,Hq,Hkv", [("qwen3", 128, 12, 3), ("qwen3", 128, 16, 2), ("gated", 256, 10, 5)])
def test_causal_key_ranges_groups(gpu_device, geo, D, Hq, Hkv):
    full = N.lib().dtree_causal_attention_workspace_bytes(D)
    assert _case(gpu_device, geo, Hq, Hkv, 700, 70, tiled=False, workspace=(full, 0), pad=128) > 0


@pytest.mark.parametrize("geo,D", [("qwen3", 128), ("gated", 256)])
@pytest.mark.parametrize("ranges,used", [(3, True), (2, True), (1, False), (0, False)])
def test_causal_short_workspace(gpu_device, geo, D, ranges, used):
    """No more ranges than the workspace holds; less than two: none."""
    size = ranges * _range_bytes(8, 2, D, 40)
    assert (_case(gpu_device, geo, 8, 2, 900, 40, workspace=(size, 0)) > 0) == used


def test_causal_misaligned_workspace_is_not_used(gpu_device):
    full = N.lib().dtree_causal_attention_workspace_bytes(128)
    assert _case(gpu_device, "qwen3", 8, 2, 900, 40, workspace=(full, 4)) == 0


@pytest.mark.parametrize("geo", ["qwen3", "gated"])
@pytest.mark.parametrize("past,n", [(0, 1), (0, 33), (0, 64), (0, 300), (1, 95), (63, 2), (64, 64), (100, 129),
                                    (1000, 31), (1985, 200)])
def test_causal_matches_float64(gpu_device, geo, past, n):
    _case(gpu_device, geo, 8, 2, past, n)


@pytest.mark.parametrize("geo,Hq,Hkv", [("qwen3", 2, 1), ("qwen3", 12, 3), ("qwen3", 16, 2), ("gated", 2, 1),
                                        ("gated", 10, 5)])
def test_causal_group_sizes(gpu_device, geo, Hq, Hkv):
    _case(gpu_device, geo, Hq, Hkv, 70, 161, tiled=False)


@pytest.mark.parametrize("geo,Hq,Hkv", [("qwen3", 4, 1), ("qwen3", 16, 2), ("gated", 4, 2)])
@pytest.mark.parametrize("past,n", [(0, 1), (130, 33), (64, 128), (70, 129)])
def test_causal_padding_workgroups(gpu_device, geo, Hq, Hkv, past, n):
    """Rows padded to 256: workgroups of padding rows alone write zeros (and
    read no page of the cache)."""
    _case(gpu_device, geo, Hq, Hkv, past, n, pad=256)


@pytest.mark.parametrize("geo", ["qwen3", "gated"])
def test_causal_without_norms(gpu_device, geo):
    _case(gpu_device, geo, 4, 2, 5, 40, norms=False)


@pytest.mark.parametrize("geo", ["qwen3", "gated"])
def test_causal_norms_at_odd_addresses(gpu_device, geo):
    _case(gpu_device, geo, 4, 2, 5, 40, norm_off=1)


def test_causal_rejects_bad_shapes(gpu_device):
    a = N.AttnArgs()
    st = torch.cuda.current_stream().cuda_stream
    assert N.lib().dtree_causal_attention(C.byref(a), 0, 1, st) == N.E_ARG  # null pointers
    t = torch.zeros(64, device=gpu_device)
    for f in ("qkv", "rope_cos", "rope_sin", "k_pages", "v_pages", "page_table", "out"):
        setattr(a, f, t.data_ptr())
    a.num_heads, a.num_kv_heads, a.head_dim, a.rows_padded, a.ld_qkv, a.ld_out = 2, 1, 64, 32, 512, 128
    assert N.lib().dtree_causal_attention(C.byref(a), 0, 1, st) == N.E_ARG  # head_dim
    a.head_dim, a.ld_out = 128, 256
    a.num_heads, a.ld_qkv = 3, 640  # a group of 3
    assert N.lib().dtree_causal_attention(C.byref(a), 0, 1, st) == N.E_ARG
    a.num_heads, a.ld_qkv = 2, 512
    for past, n in ((-1, 1), (0, 0), (0, 33)):
        assert N.lib().dtree_causal_attention(C.byref(a), past, n, st) == N.E_ARG
