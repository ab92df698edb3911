"""dtree_gdn_layer_chain's recurrence against float64 over its own q, k, v, g
and beta (the prep is checked elsewhere): both forms around their boundary,
ragged last chunks, long runs of one repeated token (equal keys, decays and
betas near 1, where powers of the chunk matrix would grow like binomials),
vanishing decays, head groups from 1 to 8, row-major outputs without padding
rows, and in every output layout an `out` buffer that holds NaN before the call
(it is scratch between the launches, and its old contents must not matter).

Bound: the recurrence is a contraction here (|k| = 1, beta and g in [0, 1]), so
fp32 rounding of a few operations per token adds up to some 2^-24 sqrt(tokens)
of the result; 2e-6 leaves a factor of ten over what was measured (2e-7).
test_chain_keeps_digits holds the sums themselves to account: y's error lies with
the dot products of 128 dims that A and U are made of (four sums 1.4e-7, one
chain 2.0e-7), the state's with what is rounded at the state's magnitude (a
chunk's update at once 2.3e-7, token by token within the chunk 3.6e-7)."""
import ctypes as C

import pytest
import torch

from dtree_hip import _native as N

pytestmark = pytest.mark.gpu


def _chain(dev, T, Hk=16, Hv=32, kind="random", rowmajor=False, h16=False, stale=False,
           y_tol=2e-6, state_tol=2e-6):
    g = torch.Generator(device=dev)
    g.manual_seed(T + Hk + 7 * Hv + len(kind))
    D = 128
    key, val = Hk * D, Hv * D
    Cd = 2 * key + val
    width = Cd + val + 2 * Hv
    rows = T if rowmajor else 32 * ((T + 31) // 32)
    rnd = lambda *s: torch.empty(*s, device=dev).normal_(generator=g)  # noqa: E731
    proj = torch.zeros(rows, (width + 63) // 64 * 64, device=dev)
    proj[:T, :width] = rnd(T, width)
    dt_bias = -4.0 + rnd(Hv)
    if kind == "repeat":  # one token over and over: keys equal once the window is full
        proj[:T, :key * 2] = proj[0, :key * 2]
        proj[:T, Cd + val:Cd + val + Hv] = 8.0          # beta ~ 1
        dt_bias = torch.full((Hv,), -12.0, device=dev)  # g ~ 1
    elif kind == "slow":  # a state that decays over thousands of tokens
        dt_bias = torch.full((Hv,), -9.0, device=dev)
    elif kind == "forget":  # g underflows to 0 for some tokens and heads
        proj[:T, Cd + val + Hv:width] *= 60.0
    win, st = rnd(3, Cd), 0.1 * rnd(Hv, D, D)
    state = st.clone()
    window = win.clone()
    z = lambda *s, dtype=torch.float32: torch.zeros(*s, dtype=dtype, device=dev)  # noqa: E731
    b = dict(q=z(rows, key), k=z(rows, key), v=z(rows, val), g=z(rows, Hv), beta=z(rows, Hv), y=z(rows, val))
    ld = val + 8 if rowmajor else val
    out = z(rows, ld, dtype=torch.float16 if h16 else torch.bfloat16)
    if stale:  # NaN as 16-bit values and as the fp32 words of the scratch
        out.view(torch.int16).fill_(-1)
    conv = torch.rand(4, Cd, device=dev, generator=g) - 0.5
    alog = torch.log(1.0 + 15.0 * torch.rand(Hv, device=dev, generator=g))
    norm = torch.ones(D, dtype=torch.bfloat16, device=dev)
    a = N.GdnArgs()
    a.rows_padded = rows; a.num_k_heads, a.num_v_heads = Hk, Hv
    a.head_k_dim = a.head_v_dim = D; a.conv_keep = 3
    a.proj = proj.data_ptr(); a.ld_proj = proj.shape[1]
    for name, t in b.items():
        setattr(a, name, t.data_ptr())
    a.window, a.state, a.out = window.data_ptr(), state.data_ptr(), out.data_ptr()
    a.conv_w, a.A_log, a.dt_bias = conv.data_ptr(), alog.data_ptr(), dt_bias.data_ptr()
    a.norm_w, a.eps = norm.data_ptr(), 1e-6
    a.out_layout, a.ld_out = (N.W_ROWMAJOR if rowmajor else N.W_TILED_F16 if h16 else N.W_TILED), ld
    print(f"gdn chain T={T} Hk={Hk} Hv={Hv} {kind} rowmajor={rowmajor} h16={h16} stale={stale}", flush=True)
    N.check(N.lib().dtree_gdn_layer_chain(C.byref(a), T, torch.cuda.current_stream().cuda_stream), "gdn chain")
    torch.cuda.synchronize()
    grp = Hv // Hk
    q, k = (b[n][:T].double().reshape(T, Hk, D).repeat_interleave(grp, 1) for n in ("q", "k"))
    v = b["v"][:T].double().reshape(T, Hv, D)
    gg, beta = b["g"][:T].double(), b["beta"][:T].double()
    S = st.double()
    y = torch.zeros(T, Hv, D, dtype=torch.float64, device=dev)
    for t in range(T):
        S = S * gg[t][:, None, None]
        d = (v[t] - (S @ k[t].unsqueeze(-1)).squeeze(-1)) * beta[t][:, None]
        S = S + d.unsqueeze(-1) * k[t].unsqueeze(1)
        y[t] = (S @ q[t].unsqueeze(-1)).squeeze(-1)
    got = b["y"][:T].double().reshape(T, Hv, D)
    assert torch.isfinite(got).all()
    ey, es = ((got - y).norm() / y.norm()).item(), ((state.double() - S).norm() / S.norm()).item()
    print(f"y {ey:.2e} state {es:.2e}", flush=True)
    assert ey <= y_tol and es <= state_tol
    assert torch.equal(window, torch.cat([win, proj[:T, :Cd]])[-3:])
    # the gated norm has replaced every scratch value in `out`
    zg = proj[:T, Cd:Cd + val].double().reshape(T, Hv, D)
    ref = y * torch.rsqrt(y.square().mean(-1, keepdim=True) + 1e-6) * zg * torch.sigmoid(zg)
    if rowmajor:
        o = out[:, :val].double().reshape(T, Hv, D)
    else:
        from dtree_hip.weights import untile_weight
        full = untile_weight(out).double()
        assert (full[T:] == 0).all()
        o = full[:T].reshape(T, Hv, D)
    # 16-bit rounding, and y's own error seen through its norm where y is small
    err = 2e-6 * y.norm() / y.norm(dim=-1, keepdim=True) * 8
    assert ((o - ref).abs() <= (2.0 ** -8 + err) * ref.abs() + 1e-5 + err).all()


@pytest.mark.parametrize("T", [40, 41, 64, 65, 79, 300])
def test_chain_forms(gpu_device, T):
    _chain(gpu_device, T)


@pytest.mark.parametrize("Hk,Hv", [(8, 16), (4, 32)])
@pytest.mark.parametrize("T", [55, 56])
def test_chain_forms_of_few_heads(gpu_device, T, Hk, Hv):
    _chain(gpu_device, T, Hk, Hv)


@pytest.mark.parametrize("kind", ["repeat", "forget"])
@pytest.mark.parametrize("T", [50, 200])
def test_chain_hard_inputs(gpu_device, T, kind):
    _chain(gpu_device, T, kind=kind)


@pytest.mark.parametrize("Hk,Hv", [(1, 1), (3, 6), (2, 16), (16, 48)])
def test_chain_head_groups(gpu_device, Hk, Hv):
    _chain(gpu_device, 77, Hk, Hv)


@pytest.mark.parametrize("T", [41, 56, 64, 65, 81])
def test_chain_row_major_unpadded(gpu_device, T):
    _chain(gpu_device, T, 2, 4, rowmajor=True)


@pytest.mark.parametrize("layout", ["tiled", "tiled_f16", "rowmajor"])
@pytest.mark.parametrize("T", [40, 41, 56, 63, 65, 81, 300])
def test_chain_ignores_old_out(gpu_device, T, layout):
    _chain(gpu_device, T, 4, 8, rowmajor=layout == "rowmajor", h16=layout == "tiled_f16", stale=True)


@pytest.mark.parametrize("kind,T,y_tol,state_tol", [("random", 300, 1.75e-7, 1.4e-7), ("slow", 1024, 3.3e-7, 3e-7)])
def test_chain_keeps_digits(gpu_device, kind, T, y_tol, state_tol):
    _chain(gpu_device, T, 4, 8, kind=kind, y_tol=y_tol, state_tol=state_tol)
