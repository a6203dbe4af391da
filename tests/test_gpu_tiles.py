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


@pytest.mark.parametrize("mesh", ["box", "hex"])
@pytest.mark.parametrize("mode", [0, 1])
def test_autotune_chooses_the_stored_factor_variant(mesh, mode):
    """The tuner chooses the variant that products from stored factors run,
    whatever the products read while it is called: from the slowest variant it
    moves to one nearer to the fastest (at 40^3 order 2 they span 81 to 143 us)."""
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    import hephaestus_amd as H
    n, p = (40, 40, 40), 2
    print(f"case autotune {mesh} mode={mode}", flush=True)
    rng = np.random.default_rng(3)
    vert = None
    if mesh == "hex":
        Z, Y, X = np.meshgrid(*[np.arange(m + 1) / m for m in n[::-1]], indexing="ij")
        vert = np.stack([X, Y, Z], -1).reshape(-1, 3) + rng.uniform(-0.001, 0.001, (X.size, 3))
    op = H.Operator(n, p, 1.0, rng.uniform(0.5, 2.0, n[0] * n[1] * n[2]), vert=vert).setup(1.0)
    x = torch.from_numpy(rng.uniform(-1, 1, op.ndofs)).cuda()
    y = torch.empty_like(x)
    op.set_factor_mode(0)
    us = {}
    for t in H.hcurl.tile_list(p):
        op.set_tile(64, *t)
        op.profile_apply(x, y, reps=5)
        us[t] = sum(op.profile_apply(x, y, reps=20).values())
    slow, fast = max(us, key=us.get), min(us.values())
    print(us, flush=True)
    assert us[slow] > 1.3 * fast
    op.set_tile(64, *slow)
    op.set_factor_mode(mode)
    y0 = op.apply(x)
    info = op.autotune(reps=10)
    assert us[op.get_tile(64)] < 0.5 * (us[slow] + fast)
    assert info["fp64_us"] > 0.0 and op.factor_mode == (mode if mesh == "box" else 0)
    if mode == 1:
        assert torch.equal(op.apply(x), y0)
    op.close()
