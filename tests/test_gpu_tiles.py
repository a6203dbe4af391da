"""Term weights of every tile variant (needs an MI355X): K x alone
(hc_op_apply_curl) equals the product of the same operator with sigma = 0 and
dt = 1, for each compiled variant, from the quadrature-point factors, on a box
and on a trilinear mesh.  A variant that ignores the weights returns (K + M) x."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mesh", ["box", "hex"])
@pytest.mark.parametrize("p", [1, 2, 3])
def test_curl_alone_every_tile(p, mesh):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    import hephaestus_amd as H
    n = (7, 5, 6)
    print(f"case curl alone p={p} {mesh}", flush=True)
    rng = np.random.default_rng(p)
    vert = None
    if mesh == "hex":
        Z, Y, X = np.meshgrid(*[np.arange(m + 1) / m for m in n[::-1]], indexing="ij")
        vert = np.stack([X, Y, Z], -1).reshape(-1, 3) + rng.uniform(-0.01, 0.01, ((n[0] + 1) * (n[1] + 1) * (n[2] + 1), 3))
    E = n[0] * n[1] * n[2]
    nu, sig = rng.uniform(0.5, 2.0, E), rng.uniform(50.0, 100.0, E)
    op = H.Operator(n, p, nu, sig, vert=vert, pec_faces=0x1A).setup(0.5)
    ref = H.Operator(n, p, nu, np.zeros(E), vert=vert, pec_faces=0x1A).setup(1.0)
    x = torch.from_numpy(rng.uniform(-1, 1, op.ndofs)).cuda()
    y = ref.set_factor_mode(0).apply(x)
    for mode in (0, 1):
        op.set_factor_mode(mode)
        for t in H.hcurl.tile_list(p):
            op.set_tile(64, *t)
            # both sides: rounding of a few units of 2^-53 (the tile kernels are within 3e-15 of 64-bit references)
            assert float((op.apply_curl(x) - y).norm()) <= 2e-14 * float(y.norm()), (mode, t)
    op.close()
    ref.close()
