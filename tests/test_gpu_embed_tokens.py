"""dtree_embed_tokens over widths that do not fill a workgroup's 128 columns,
ragged row counts and out-of-range tokens: x is the embedding row exactly (zero
past n), xg its product with the norm weight (one 16-bit rounding, with the low
plane two), ss the sums of squares of 32 columns (fp32 sums of 32 terms)."""
import pytest
import torch

from dtree_hip import _native as N
from dtree_hip.weights import tile_weight, tile_weight_f16, untile_weight

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H", [64, 192, 320, 2560])
@pytest.mark.parametrize("rows,n", [(32, 1), (96, 96), (160, 130)])
@pytest.mark.parametrize("layout", [N.W_ROWMAJOR, N.W_TILED, N.W_TILED_F16])
def test_embed_tokens(gpu_device, H, rows, n, layout):
    V = 320
    g = torch.Generator(device=gpu_device)
    g.manual_seed(H + rows)
    emb = torch.empty(V, H, device=gpu_device).normal_(generator=g).to(torch.bfloat16)
    w = (1 + 0.1 * torch.empty(H, device=gpu_device).normal_(generator=g)).to(torch.bfloat16)
    tok = torch.randint(0, V, (n,), generator=g, device=gpu_device, dtype=torch.int32)
    tok[n // 2] = V if n > 1 else tok[n // 2]  # out of range: a zero row
    f16 = layout == N.W_TILED_F16
    table = emb if layout == N.W_ROWMAJOR else tile_weight_f16(emb.half()) if f16 else tile_weight(emb)
    dt = torch.float16 if f16 else torch.bfloat16
    x = torch.full((rows, H), 5.0, device=gpu_device)
    xg = torch.full((2, rows, H), 5.0, dtype=dt, device=gpu_device)
    ss = torch.full((rows // 32, H // 32, 32), 5.0, device=gpu_device)
    N.call("dtree_embed_tokens", tok.data_ptr(), n, table.data_ptr(), layout, None, V, H, w.data_ptr(), rows,
           x.data_ptr(), xg[0].data_ptr(), None if f16 else xg[1].data_ptr(), layout, ss.data_ptr(),
           torch.cuda.current_stream().cuda_stream)
    ref = torch.zeros(rows, H, dtype=torch.float64, device=gpu_device)
    ok = tok < V
    ref[:n][ok] = (emb.half() if f16 else emb)[tok[ok].long()].double()
    assert torch.equal(x.double(), ref)
    y = ref * w.double()
    planes = [t if layout == N.W_ROWMAJOR else untile_weight(t) for t in xg]
    got = planes[0].double() + (0.0 if f16 else planes[1].double())
    assert ((got - y).abs() <= 2.0 ** (-11 if f16 else -16) * y.abs() + 2.0 ** -24).all()
    sq = ref.square().reshape(rows // 32, 32, H // 32, 32).sum(-1).transpose(1, 2)
    assert ((ss.double() - sq).abs() <= 32 * 2.0 ** -24 * sq).all()
