"""dtree_gemm_long's tile shapes against a float64 product.

The fp16 path picks one of eight tile shapes by rows and columns, the q4 path
one of four; each case names the tile it is for, which the library has to
confirm, and test_every_tile_has_a_case that none is left out: with ragged last
row and column tiles, with fewer K stages than the pipeline holds, and with
outputs too misaligned for the vector stores. Bounds: the fp32 accumulation of K products differs from
the exact sum by at most K 2^-24 sum |x w| (checked in the result's units);
fp16 and bf16 outputs add their own rounding (2^-11, 2^-8 relative)."""
import ctypes as C

import pytest
import torch

from dtree_hip import _native as N
from dtree_hip.weights import q4_dequant, q4_random_mlx, q4_to_tiled, Q4Linear, tile_weight, tile_weight_f16, untile_weight

pytestmark = pytest.mark.gpu


def _silu(t):
    return t * torch.sigmoid(t)


def _tile(rows, n, k, epi, w_layout, pair=False):
    a = N.GemmArgs()
    a.rows_padded, a.n, a.k, a.epilogue, a.w_layout, a.x_lo = rows, n, k, epi, w_layout, 16 if pair else None
    t = N.lib().dtree_gemm_long_tile(C.byref(a))
    return t // 1000, t % 1000


def _long(dev, rows, n, k, epi, misaligned=False, seed=0, form="f16", tile=None):
    """form: fp16 operands, bf16 operands, or bf16 weights with the activations
    and the outputs as split pairs of bf16 planes (value = hi + lo); q4 weights
    with bf16 activations."""
    g = torch.Generator(device=dev)
    g.manual_seed(seed + rows + 3 * n + 7 * k)
    h16, pair, q4 = form == "f16", form == "pair", form == "q4"
    dt = torch.float16 if h16 else torch.bfloat16
    x = torch.empty(rows, k, device=dev).normal_(generator=g)
    xl = (x - x.to(dt).float()).to(dt)
    x = x.to(dt)
    w = torch.empty(n, k, device=dev).normal_(0.0, 0.05, generator=g).to(dt)
    to_tiles = tile_weight_f16 if h16 else tile_weight
    xt, xlt, wt = to_tiles(x), to_tiles(xl), to_tiles(w)
    layout = N.W_TILED_F16 if h16 else N.W_TILED
    off = 1 if misaligned else 0  # rows of odd length from an odd element: no vector access is aligned
    width = n // 2 if epi == N.EPI_SWIGLU else n
    ld = width + off
    a = N.GemmArgs()
    a.x = xt.data_ptr(); a.w = wt.data_ptr(); a.x_layout = a.w_layout = layout
    if pair:
        a.x_lo = xlt.data_ptr()
        x = x.double() + xl.double()
    if q4:
        wq, sc, bi = q4_random_mlx(n, k, g, dev)
        lin = Q4Linear(*q4_to_tiled(wq, sc, bi))
        a.w, a.w_scales, a.w_layout = lin.words.data_ptr(), lin.sb.data_ptr(), N.W_Q4G64
        w = q4_dequant(lin)
    if tile is not None:
        assert _tile(rows, n, k, epi, a.w_layout, pair) == tile
    a.ldx = k; a.rows_padded = rows; a.n = n; a.k = k; a.epilogue = epi
    a.norm_dim = k; a.eps = 1e-6
    a.out_layout = N.W_ROWMAJOR if misaligned else layout
    f32 = torch.zeros(rows * (n + off) + off, device=dev).normal_(generator=g)
    res0 = f32[off:].view(rows, n + off)[:, :n].double().clone()
    act, actl = (torch.zeros(rows * ld + off, dtype=torch.int16, device=dev) for _ in range(2))
    hid = torch.zeros(rows * (n + off) + off, dtype=torch.bfloat16, device=dev)
    norm = (1 + 0.1 * torch.empty(n, device=dev).normal_(generator=g)).to(torch.bfloat16)
    ss = torch.rand(rows // 32, k // 32, 32, device=dev, generator=g) + 0.5
    sso = torch.zeros(rows // 32, n // 32, 32, device=dev)
    a.out_f32 = f32.data_ptr() + 4 * off; a.ld_out_f32 = n + off
    a.out_bf16 = act.data_ptr() + 2 * off; a.ld_out_bf16 = ld
    if pair:
        a.out_lo = actl.data_ptr() + 2 * off
    rs = torch.ones(rows, dtype=torch.float64, device=dev)
    if epi == N.EPI_RESIDUAL:
        a.next_norm = norm.data_ptr(); a.ss_out = sso.data_ptr()
        a.hidden_out = hid.data_ptr() + 2 * off; a.ld_hidden = n + off
    else:
        a.ss_in = ss.data_ptr(); a.ss_tiles = k // 32
        rs = torch.rsqrt(ss.double().transpose(1, 2).reshape(rows, -1).sum(1) / k + 1e-6)
    print(f"gemm_long rows={rows} n={n} k={k} epi={epi} misaligned={misaligned} {form}", flush=True)
    N.check(N.lib().dtree_gemm_long(C.byref(a), torch.cuda.current_stream().cuda_stream), "gemm_long")
    torch.cuda.synchronize()
    acc = x.double() @ w.double().T
    # (q4: the bias term stands apart from the group sums, on values up to 31 |s|)
    mag = (31 * sc.double().abs() + bi.double().abs()).repeat_interleave(64, 1) * 2 if q4 else w.double().abs()
    bound = (x.double().abs() @ mag.T).max().item() * k * 2.0 ** -24 * rs.max().item() + 1e-6
    f = f32[off:].view(rows, n + off)[:, :n].double()
    if misaligned:  # row-major bf16
        b = sum(t[off:].view(rows, ld)[:, :width].view(torch.bfloat16).double() for t in (act, actl))
    else:
        b = sum(untile_weight(t.view(dt).view(rows, width)).double() for t in (act, actl))
    # (each plane of a pair rounds what it is given by 2^-8 at most)
    rnd = 2.0 ** -16 if pair else 2.0 ** -11 if h16 and not misaligned else 2.0 ** -8
    if epi == N.EPI_STORE_F32:
        assert (f - acc * rs[:, None]).abs().max().item() <= bound
    elif epi == N.EPI_STORE_BF16:
        ref = acc * rs[:, None]
        assert ((b - ref).abs() <= bound + rnd * ref.abs() + 2.0 ** -24).all()
    elif epi == N.EPI_SWIGLU:
        v = (acc * rs[:, None]).reshape(rows, n // 32, 2, 16)
        ga, up = v[:, :, 0].reshape(rows, -1), v[:, :, 1].reshape(rows, -1)
        ref = _silu(ga) * up
        # |silu'| <= 1.1; the device's exp and divide are within a few ulp
        err = bound * (1.1 * up.abs() + ga.abs()) + 1e-6 * ref.abs()
        assert ((b - ref).abs() <= err + rnd * ref.abs() + 2.0 ** -24).all()
    else:
        ref = res0 + acc
        assert (f - ref).abs().max().item() <= bound + 2.0 ** -23 * ref.abs().max().item()
        xg = f * norm.double()
        assert ((b - xg).abs() <= (rnd + 1e-6) * xg.abs() + 2.0 ** -24).all()
        h = hid[off:].view(rows, n + off)[:, :n]
        assert torch.equal(h, f.float().to(torch.bfloat16))
        want = f.square().reshape(rows // 32, 32, n // 32, 32).sum(-1).transpose(1, 2)
        torch.testing.assert_close(sso.double(), want, rtol=1e-5, atol=1e-5)


# (rows, n, tile, tile with the residual epilogue, which the two widest do not take)
SHAPES = [(128, 256, (64, 64), (64, 64)), (128, 6144, (64, 64), (64, 64)), (384, 2560, (64, 64), (64, 64)),
          (640, 2432, (64, 128), (64, 128)), (256, 6144, (64, 128), (64, 128)),
          (896, 2432, (128, 128), (128, 128)), (256, 12288, (128, 128), (128, 128)),
          (384, 12288, (256, 128), (256, 128)), (768, 6144, (256, 128), (256, 128)),
          (384, 19456, (256, 192), (256, 192)), (768, 12288, (256, 192), (256, 192)),
          (640, 19456, (256, 256), (256, 256)), (896, 12416, (256, 256), (256, 256)),
          (384, 6144, (128, 128), (128, 128)), (768, 2560, (64, 128), (64, 128)),
          (1152, 6144, (256, 128), (256, 128)), (1152, 12416, (256, 256), (256, 256)), (1152, 24576, (256, 256), (256, 256)),
          (640, 24576, (256, 320), (256, 192)), (1024, 19456, (256, 320), (256, 192)),
          (1152, 19456, (256, 384), (256, 192)), (1024, 24576, (256, 384), (256, 192))]


@pytest.mark.parametrize("rows,n,tile,tile_res", SHAPES)
@pytest.mark.parametrize("epi", [N.EPI_STORE_F32, N.EPI_RESIDUAL, N.EPI_SWIGLU, N.EPI_STORE_BF16])
@pytest.mark.parametrize("k", [64, 320])
def test_long_tiles_match_float64(gpu_device, rows, n, tile, tile_res, epi, k):
    _long(gpu_device, rows, n, k, epi, tile=tile_res if epi == N.EPI_RESIDUAL else tile)


# bf16 weights, with one and two activation planes: 128x128 tiles, several per
# CU and a K loop shorter and longer than the pipeline
@pytest.mark.parametrize("form", ["bf16", "pair"])
@pytest.mark.parametrize("rows,n,k", [(128, 256, 64), (384, 384, 128), (640, 512, 320), (1152, 6144, 192)])
@pytest.mark.parametrize("epi", [N.EPI_STORE_F32, N.EPI_RESIDUAL, N.EPI_SWIGLU, N.EPI_STORE_BF16])
@pytest.mark.parametrize("misaligned", [False, True])
def test_long_bf16_matches_float64(gpu_device, rows, n, k, epi, form, misaligned):
    _long(gpu_device, rows, n, k, epi, misaligned=misaligned, form=form)


@pytest.mark.parametrize("form", ["bf16", "pair"])
def test_long_bf16_64_column_tail(gpu_device, form):
    _long(gpu_device, 256, 448, 192, N.EPI_STORE_F32, form=form)


TAILS = [(128, 64, (64, 64)), (128, 12352, (64, 128)), (640, 4160, (128, 128)), (384, 12352, (256, 128)),
         (384, 16448, (256, 192)), (1024, 12352, (256, 256)), (640, 21824, (256, 320)), (1152, 19520, (256, 384)), (640, 19520, (256, 256)),
         (1024, 19520, (256, 320)), (1152, 24640, (256, 256))]


@pytest.mark.parametrize("rows,n,tile", TAILS)
def test_long_tiles_64_column_tail(gpu_device, rows, n, tile):
    _long(gpu_device, rows, n, 192, N.EPI_STORE_F32, tile=tile)


@pytest.mark.parametrize("rows,n", [(384, 256), (1152, 6144), (1024, 19456), (1152, 19456)])
@pytest.mark.parametrize("epi", [N.EPI_STORE_F32, N.EPI_RESIDUAL, N.EPI_SWIGLU, N.EPI_STORE_BF16])
def test_long_tiles_misaligned_outputs(gpu_device, rows, n, epi):
    _long(gpu_device, rows, n, 128, epi, misaligned=True)


# Ragged last row and column tiles; k % 128 != 0 keeps to the three wider tiles.
# A K of 5, 8, 9 and 19 groups ends inside, at and past the eight groups of a
# correction step.
Q4_SHAPES = [(128, 256, 640, (128, 128)), (128, 512, 512, (128, 128)), (384, 384, 1152, (128, 128)),
             (384, 12416, 512, (128, 256)), (128, 256, 320, (128, 256)), (256, 384, 1216, (128, 256)),
             (1152, 9728, 512, (256, 192)), (384, 24576, 576, (256, 192)),
             (384, 19456, 320, (128, 256)), (640, 19456, 576, (256, 256)), (1152, 12416, 1152, (256, 256))]
Q4_TAILS = [(640, 19520, 576, (256, 256)), (1152, 12352, 512, (256, 256)),
            (256, 320, 1216, (128, 256)), (384, 21824, 512, (256, 192)), (1152, 12352, 1216, (256, 256))]


@pytest.mark.parametrize("rows,n,k,tile", Q4_SHAPES)
@pytest.mark.parametrize("epi", [N.EPI_RESIDUAL, N.EPI_SWIGLU, N.EPI_STORE_BF16])
def test_long_q4_epilogues(gpu_device, rows, n, k, tile, epi):
    _long(gpu_device, rows, n, k, epi, form="q4", tile=tile)


@pytest.mark.parametrize("rows,n", [(256, 384), (1152, 9728)])
@pytest.mark.parametrize("epi", [N.EPI_STORE_F32, N.EPI_RESIDUAL, N.EPI_SWIGLU, N.EPI_STORE_BF16])
def test_long_q4_misaligned_outputs(gpu_device, rows, n, epi):
    _long(gpu_device, rows, n, 320, epi, misaligned=True, form="q4")


@pytest.mark.parametrize("rows,n,k,tile", Q4_SHAPES + Q4_TAILS)
@pytest.mark.parametrize("lo", [False, True])
@pytest.mark.parametrize("mean", [0.0, 4.0])
def test_long_q4_tiles_match_float64(gpu_device, rows, n, k, tile, lo, mean):
    """fp32 store; weights with a constant-group (scale 0) row block and a group
    whose bias dwarfs its scale; activations with and without a mean. The group
    sums are exact products of bf16 values, at most 31 |s| per unit of |x|,
    accumulated in fp32, and the bias term carries 24 bits, so the error stays
    within k 2^-23 of sum |x| (|s| 31 + |b|). Its norm: a rounding of the
    accumulator is 0.29 * 2^-24 of it at random, there are k / 64 of them, and
    its rms is that of up to eight groups of 16 + q, (16 + 7.5) / 4.6 times the
    result's share of eight groups: 5.1 sqrt(8) 0.29 2^-24 = 2.5e-7 of the
    result, and as much again at the most for the sums inside the groups and the
    result itself. (Nibbles as 128 + q gave 4.4e-7 to 1.6e-6.)"""
    g = torch.Generator(device=gpu_device)
    g.manual_seed(rows + n + k)
    wq, sc, bi = q4_random_mlx(n, k, g, gpu_device)
    sc[:32, 0] = 0.0
    bi[32:64, 1] = 40.0
    lin = Q4Linear(*q4_to_tiled(wq, sc, bi))
    xf = torch.empty(rows, k, device=gpu_device).normal_(mean, 1.0, generator=g)
    hi = xf.to(torch.bfloat16)
    low = (xf - hi.float()).to(torch.bfloat16)
    xt, xlt = tile_weight(hi), tile_weight(low)
    ss = torch.rand(rows // 32, k // 32, 32, device=gpu_device, generator=g) + 0.5
    out = torch.zeros(rows, n, device=gpu_device)
    a = N.GemmArgs()
    a.x = xt.data_ptr(); a.x_lo = xlt.data_ptr() if lo else None
    a.x_layout = N.W_TILED; a.ldx = k; a.rows_padded = rows
    a.w = lin.words.data_ptr(); a.w_scales = lin.sb.data_ptr(); a.w_layout = N.W_Q4G64; a.n = n; a.k = k
    a.epilogue = N.EPI_STORE_F32; a.out_f32 = out.data_ptr(); a.ld_out_f32 = n
    a.ss_in = ss.data_ptr(); a.ss_tiles = k // 32; a.norm_dim = k; a.eps = 1e-6
    assert _tile(rows, n, k, N.EPI_STORE_F32, N.W_Q4G64, lo) == ((128, 128) if lo else tile)
    print(f"q4 gemm_long rows={rows} n={n} k={k} lo={lo} mean={mean}", flush=True)
    N.check(N.lib().dtree_gemm_long(C.byref(a), torch.cuda.current_stream().cuda_stream), "gemm_long")
    torch.cuda.synchronize()
    rs = torch.rsqrt(ss.double().transpose(1, 2).reshape(rows, -1).sum(1) / k + 1e-6)
    x = hi.double() + (low.double() if lo else 0.0)
    ref = (x @ q4_dequant(lin).double().T) * rs[:, None]
    mag = (x.abs() @ (31.0 * sc.double().abs() + bi.double().abs()).repeat_interleave(64, 1).T) * rs[:, None]
    assert ((out.double() - ref).abs() <= k * 2.0 ** -23 * mag).all()
    # (without the columns of the large bias, whose results would hide the others')
    keep = torch.arange(n, device=gpu_device) // 32 != 1
    rel = ((out.double() - ref)[:, keep].norm() / ref[:, keep].norm()).item()
    print(f"relative error {rel:.2e}", flush=True)
    assert rel <= 4e-7, rel  # measured below 3e-7
