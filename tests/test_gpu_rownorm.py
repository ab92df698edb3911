"""dtree_rownorm against float64: rows, widths and statistics tiles that do not
fill a workgroup or a wave, and operands that rule the vector accesses out. The
statistics are random sums (not those of x), so their layout is checked too. A
result is the bf16 rounding of a few fp32 roundings: within 2^-8 relative."""
import pytest
import torch

from dtree_hip import _native as N

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 32, 96, 128])
@pytest.mark.parametrize("H,tiles,pad,off", [(64, 2, 0, 0), (2560, 80, 0, 0), (4096, 128, 4, 0), (1030, 33, 1, 0),
                                             (1028, 65, 0, 1), (3, 1, 2, 0)])
def test_rownorm(gpu_device, rows, H, tiles, pad, off):
    g = torch.Generator(device=gpu_device)
    g.manual_seed(rows + H)
    ld = H + pad
    x = torch.empty(off + rows * ld, device=gpu_device).normal_(generator=g)[off:].view(rows, ld)
    blocks = (rows + 31) // 32
    ss = torch.empty(blocks, tiles, 32, device=gpu_device).uniform_(0.5, 2.0, generator=g)
    w = (1 + 0.1 * torch.empty(H, device=gpu_device).normal_(generator=g)).to(torch.bfloat16)
    out = torch.full((rows * ld + off,), 7.0, dtype=torch.bfloat16, device=gpu_device)[off:].view(rows, ld)
    st = torch.cuda.current_stream().cuda_stream
    N.call("dtree_rownorm", x.data_ptr(), ld, rows, H, ss.data_ptr(), tiles, w.data_ptr(), 1e-6, out.data_ptr(), ld, st)
    tot = ss.double().sum(1).reshape(-1)[:rows]
    ref = x[:, :H].double() * torch.rsqrt(tot / H + 1e-6)[:, None] * w.double()
    assert ((out[:, :H].double() - ref).abs() <= 2.0 ** -8 * ref.abs()).all()
    assert (out[:, H:] == 7.0).all()
