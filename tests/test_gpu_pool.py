"""The pool in pieces of 8 channels, with and without the copy into a
concatenation buffer, at channel counts and box sizes beside those it takes:
sums of eight bf16 values in the order of the window, so exact."""
import pytest
import torch

from nga2_amd import unet

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(2, 2, 2), (6, 4, 10), (34, 18, 6), (7, 5, 3)])
@pytest.mark.parametrize("c", [8, 32, 12])
def test_pool_and_copy(dims, c):
    nx, ny, nz = dims
    print(f"\n[pool {dims} {c}]", flush=True)
    L = unet.lib()
    gen = torch.Generator(device="cuda").manual_seed(4)
    x = torch.randn((nz, ny, nx, c), device="cuda", generator=gen).to(torch.bfloat16)
    ctot, d0 = 2 * c + 8, c + 8 if c % 8 == 0 else 4
    m = [n // 2 for n in dims]
    out = torch.empty((m[2], m[1], m[0], c), dtype=torch.bfloat16, device="cuda")
    out2 = torch.empty_like(out)
    cat = torch.full((nz, ny, nx, ctot), 3.0, dtype=torch.bfloat16, device="cuda")
    torch.cuda.synchronize()
    assert L.ngapnet_pool2(x.data_ptr(), out.data_ptr(), nx, ny, nz, c, None) == 0
    assert L.ngapnet_pool2_cat(x.data_ptr(), out2.data_ptr(), cat.data_ptr(), nx, ny, nz, c, ctot, d0, None) == 0
    torch.cuda.synchronize()
    w = x[: 2 * m[2], : 2 * m[1], : 2 * m[0]].float()
    s = torch.zeros((m[2], m[1], m[0], c), device="cuda")
    for q in range(8):
        s += w[q >> 2 :: 2, (q >> 1) & 1 :: 2, q & 1 :: 2]
    want = (0.125 * s).to(torch.bfloat16)
    assert torch.equal(out, want) and torch.equal(out2, want)
    assert torch.equal(cat[..., d0 : d0 + c], x)
    rest = torch.cat([cat[..., :d0], cat[..., d0 + c :]], -1)
    assert (rest == 3.0).all()
