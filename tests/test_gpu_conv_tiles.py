"""The tiled BF16 convolution kernels at the edges of their tiles and ranges:
one tile, workgroups that walk over several tiles and channel chunks, rows that
are a multiple of 16 but not of 32, columns cut into ranges of planes, and
output pointers that allow no vector stores.

Reference: float64 products of the same BF16 values, tap by tap. The kernels
accumulate n = 27 cin (forward) or n = voxels (weight gradient) products in
FP32, in an order of their own: an error of a few sqrt(n) 2^-24 of the sums'
scale. The bounds of test_gpu_unet.py (2e-6 and 2e-5 of max|ref|) hold at these
sizes as well. BF16 outputs are within one rounding (2^-8) of the reference.
"""
import ctypes as C

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"

SHAPES = [
    ((16, 4, 4), 32, 32),    # one tile
    ((16, 4, 8), 64, 32),    # two tiles, two channel chunks
    ((48, 12, 4), 32, 64),   # rows of 48: the K = 16 weight gradient; 12 rows: no 8-row tiles
    ((32, 4, 20), 64, 64),   # one column of 32 voxels, planes cut unevenly
    ((64, 64, 64), 32, 64),  # 1024 8-row tiles: workgroups walk over two each
    ((128, 40, 20), 64, 32),  # 8-row tiles, ragged share per workgroup
]


def _off(tap):
    return tap % 3 - 1, (tap // 3) % 3 - 1, tap // 9 - 1


def _shifted(x, shape, tap):
    dx, dy, dz = _off(tap)
    g = x.reshape(shape[2], shape[1], shape[0], -1)
    return torch.roll(g, (-dz, -dy, -dx), (0, 1, 2)).reshape(x.shape)


def _p(t):
    return C.c_void_p(t.data_ptr())


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("shape,cin,cout", SHAPES)
def test_forward_and_weight_gradient(shape, cin, cout, shift):
    from nga2_amd import unet

    L = unet.lib()
    print(f"\n[conv tiles {shape} {cin}->{cout} shift {shift}]", flush=True)
    gen = torch.Generator(device=DEV).manual_seed(7)
    V = shape[0] * shape[1] * shape[2]
    x = torch.randn(V, cin, generator=gen, device=DEV).to(torch.bfloat16)
    w = (torch.randn(27, cout, cin, generator=gen, device=DEV) / (27 * cin) ** 0.5).to(torch.bfloat16)
    g = torch.randn(V, cout, generator=gen, device=DEV).to(torch.bfloat16)
    out = torch.zeros(V * cout + 1, device=DEV)[shift:shift + V * cout]
    outb = torch.zeros(V * cout + 1, dtype=torch.bfloat16, device=DEV)[shift:shift + V * cout]
    parts = L.ngapnet_wgrad_parts(*shape, cin, cout)
    part = torch.zeros(parts * 27 * cin * cout + 1, device=DEV)[shift:]
    dw = torch.zeros(27 * cin * cout + 1, device=DEV)[shift:shift + 27 * cin * cout]
    unet._enter()
    rc = L.ngapnet_conv3_fwd(_p(x), _p(w), _p(out), _p(outb), *shape, cin, cout, 1, None)
    rc |= L.ngapnet_conv3_wgrad(_p(x), _p(g), _p(dw), _p(part), *shape, cin, cout, None)
    unet._leave()
    assert rc == 0
    x64, w64, g64 = x.double(), w.double(), g.double()
    ref = sum(_shifted(x64, shape, t) @ w64[t].T for t in range(27))
    err = (out.double().reshape(V, cout) - ref).abs().max() / ref.abs().max()
    assert float(err) <= 2e-6, float(err)
    relu = torch.relu(ref)
    lim = relu * 2.0 ** -8 + 2e-6 * ref.abs().max()
    assert bool(((outb.double().reshape(V, cout) - relu).abs() <= lim).all())
    dref = torch.stack([g64.T @ _shifted(x64, shape, t) for t in range(27)])
    err = (dw.double().reshape(27, cout, cin) - dref).abs().max() / dref.abs().max()
    assert float(err) <= 2e-5, float(err)


@pytest.mark.parametrize("shape,cin", [((16, 4, 4), 32), ((16, 4, 8), 96), ((64, 64, 64), 64)])
def test_forward_sums_in_order(shape, cin):
    """An output sums its taps in FP32 by channel chunk, dz, dy, dx: another
    order would round elsewhere and, through BF16 outputs, change a network's
    results. One weight of each (chunk, tap) is +-2^24 or +-1 and the input is
    1, so that every tap adds one number and the sum depends on the order."""
    from nga2_amd import unet

    L = unet.lib()
    print(f"\n[conv order {shape} {cin}]", flush=True)
    cout, chunks = 32, cin // 32
    gen = torch.Generator(device="cpu").manual_seed(11)
    val = torch.tensor([2.0 ** 24, -(2.0 ** 24), 1.0, -1.0])[torch.randint(4, (chunks, 27, cout), generator=gen)]
    at = torch.randint(32, (chunks, 27, cout, 1), generator=gen)
    w = torch.zeros(chunks, 27, cout, 32).scatter_(3, at, val[..., None])
    w = w.permute(1, 2, 0, 3).reshape(27, cout, cin).to(torch.bfloat16).contiguous().to(DEV)
    want = torch.zeros(cout)
    for c in range(chunks):
        for t in range(27):
            want = want + val[c, t]
    assert not torch.equal(want, val.double().sum((0, 1)).float())
    V = shape[0] * shape[1] * shape[2]
    x = torch.ones(V, cin, dtype=torch.bfloat16, device=DEV)
    out = torch.zeros(V, cout, device=DEV)
    unet._enter()
    rc = L.ngapnet_conv3_fwd(_p(x), _p(w), _p(out), None, *shape, cin, cout, 0, None)
    unet._leave()
    assert rc == 0
    assert torch.equal(out.cpu(), want.expand(V, cout))


@pytest.mark.parametrize("n,cin,cout", [((64, 64, 64), 128, 128), ((32, 32, 32), 256, 256), ((128, 128, 128), 96, 32)])
def test_weight_gradient_sums_stay_short(n, cin, cout):
    """Many channel blocks leave few workgroups per block; the sums of each must
    not get longer for it. n additions of terms of random sign leave an error of
    0.41 x 2^-24 of the sum at each, 2^-24 sqrt(n / 12) in all; the matrix unit's
    own additions round worse (measured: sqrt(n / 4)). The bound is that of L
    products of 32 voxels each in at most 256 partials, and their sum one by
    one, with n / 8 and L / 3.5 for margin."""
    from nga2_amd import unet

    L = unet.lib()
    print(f"\n[conv wgrad sums {n} {cin}->{cout}]", flush=True)
    gen = torch.Generator(device=DEV).manual_seed(5)
    V = n[0] * n[1] * n[2]
    x = torch.relu(torch.randn(V, cin, generator=gen, device=DEV)).to(torch.bfloat16)
    g = torch.randn(V, cout, generator=gen, device=DEV).to(torch.bfloat16)
    G = L.ngapnet_wgrad_parts(*n, cin, cout)
    part = torch.empty(G * 27 * cin * cout, device=DEV)
    dw = torch.empty(27, cout, cin, device=DEV)
    unet._enter()
    rc = L.ngapnet_conv3_wgrad(_p(x), _p(g), _p(dw), _p(part), *n, cin, cout, None)
    unet._leave()
    assert rc == 0
    x64, gt = x.double(), g.double().T.contiguous()
    num = den = 0.0
    for t in range(27):
        ref = gt @ _shifted(x64, n, t)
        num += float((dw[t].double() - ref).square().sum())
        den += float(ref.square().sum())
    err = (num / den) ** 0.5
    lim = 2.0 ** -24 * (V / 32 / G / 3.5 + G / 8) ** 0.5
    print(f"error {err:.2e}, bound {lim:.2e}", flush=True)
    assert err <= lim


def test_planes_beyond_4_gib():
    """Planes of 4 GiB and more take 64-bit offsets. The input repeats a smaller
    box 12 times in y, so the output repeats that box's, bit for bit; an offset
    that wrapped at 2^32 bytes would be 8192 rows off, no multiple of the box."""
    from nga2_amd import unet

    L = unet.lib()
    nx, ny, nz, c, reps = 8192, 684, 4, 32, 12
    assert nx * ny * reps * c * 2 >= 2 ** 32 and 2 ** 32 // (nx * c * 2) % ny != 0
    print("\n[conv planes beyond 4 GiB]", flush=True)
    gen = torch.Generator(device=DEV).manual_seed(3)
    x = torch.randn(nz, 1, ny, nx * c, generator=gen, device=DEV).to(torch.bfloat16)
    w = (torch.randn(27, c, c, generator=gen, device=DEV) / (27 * c) ** 0.5).to(torch.bfloat16)
    want = torch.empty_like(x)
    big = x.expand(nz, reps, ny, nx * c).contiguous()
    got = torch.empty_like(big)
    unet._enter()
    rc = L.ngapnet_conv3_fwd(_p(x), _p(w), None, _p(want), nx, ny, nz, c, c, 1, None)
    rc |= L.ngapnet_conv3_fwd(_p(big), _p(w), None, _p(got), nx, ny * reps, nz, c, c, 1, None)
    unet._leave()
    assert rc == 0
    assert float(want.float().abs().max()) > 0
    for r in range(reps):
        assert torch.equal(got[:, r], want[:, 0]), r
    del big, got
    torch.cuda.empty_cache()
