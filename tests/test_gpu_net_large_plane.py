"""The network on a plane of more than 2^27 points, whose 16-channel
activations have more than 2^31 elements: places of the plane's last rows
equal the same input as a small box of its own, bit for bit, away from the box
edges (the three 3^3 layers reach three points)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_plane_beyond_32_bit_offsets(torch_cuda):
    import pamr_amrd_amd as pm
    torch = torch_cuda
    ny, nx, m = 8269, 16411, 70
    assert nx * (ny - m) * 16 > 2 ** 31
    print(f"case network plane {nx} x {ny}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn((1, ny, nx), generator=gen, device="cuda")
    net = pm.Net(seed=3)
    y = torch.full_like(x, float("nan"))
    net.infer(x, y, (1, ny, nx))
    for j0, i0 in ((ny - m, nx - m), (ny - m, 0), (0, nx - m), (ny // 2, nx // 2)):
        xs = x[:, j0:j0 + m, i0:i0 + m].contiguous()
        ys = torch.empty_like(xs)
        net.infer(xs, ys, (1, m, m))
        at_j, at_i = slice(0 if j0 == 0 else 3, m if j0 + m == ny else m - 3), slice(0 if i0 == 0 else 3, m if i0 + m == nx else m - 3)
        assert torch.equal(y[:, j0:j0 + m, i0:i0 + m][:, at_j, at_i], ys[:, at_j, at_i]), (j0, i0)
    assert np.isfinite(y[0, -1].cpu().numpy()).all()
