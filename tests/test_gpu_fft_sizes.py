"""The FFT convolution at every size with a specialised form (and next to
them), through the PM force meshes, against the FP64 model.

Tolerance: white-noise density, so the force meshes carry FP32 rounding of
about log2(n^3) butterflies, eps/2 * sqrt(3 log2 n) < 3e-7, times at most 4
for the difference stencil's cancellation at the smallest scales: 1.2e-6,
taken as 2e-6."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from cube_nu_amd import pmdiff  # noqa: E402
from oracle import pm_torch as ref  # noqa: E402

PLANES = [16, 24, 32, 40, 48, 56, 64, 72, 80, 88, 96, 104, 112, 120, 128, 144, 160, 168, 176, 192]
EVEN = [18, 20, 22, 26, 28, 30, 36, 42, 44, 50, 52, 54, 60, 66, 70, 78, 84, 90, 98, 100, 108, 110, 126, 130, 132, 140,
        150, 154, 156, 162, 180, 182, 196, 198]  # the other even sizes of the plane form
LINES = [208, 210, 216, 224, 234, 240, 252, 256, 288]
GENERIC = [200, 220, 242, 250]


@pytest.mark.gpu
@pytest.mark.parametrize("n,batch", [(n, 2 if n <= 128 else 1) for n in PLANES + EVEN + LINES + GENERIC]
                         + [(n, 512) for n in (16, 24, 32)])  # many small cubes: one workgroup each
def test_gpu_force_meshes_every_fft_size(n, batch):
    B = batch
    pm = pmdiff.PMForce(n, B, 1.0)
    G = torch.from_numpy(pm.green().astype(np.float64)).cuda()
    gen = torch.Generator(device="cuda").manual_seed(n)
    np_ = min(n ** 3 // 4, 200006 // B)
    x = torch.rand((B * np_, 3), generator=gen, device="cuda") * n
    _, F = pm.force(x)
    want = ref.fd_force(ref.potential(ref.deposit(x.double(), B, n), G))
    err = float(torch.linalg.vector_norm(F.double() - want) / torch.linalg.vector_norm(want))
    print(f"n={n} F rel {err:.2e}")
    assert err <= 2e-6
    pm.close()
