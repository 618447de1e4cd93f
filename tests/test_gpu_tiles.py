"""Every tile of the 1-bit LDS-DMA product (csrc/ob_gemm2.h: 256 rows x 128 / 112 / 96 tokens, 128 rows x 128 / 96), whole and in K slices, at the edges of the tiles.

An output is the same chain of products in every tile, so whole products have the same bits; K slices add up to four of its pieces.  The tile is read once per
process (OB_GEMM3_RT, OB_GEMM3_KSPLIT)."""
import os
import subprocess
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CHILD = """
import sys
import numpy as np, torch
from torch import nn
from onebit_amd import BitLinearInf
out = {}
for T in (65, 96, 97, 128, 129, 225, 257):
    for K, N in ((1024, 256), (1280, 260), (2048, 1000), (2816, 2824)):
        g = torch.Generator(device="cuda").manual_seed(T * 7 + K)
        m = BitLinearInf(K, N, device="cuda", dtype=torch.float16)
        m.weight.data = torch.randint(0, 256, (N, K // 8), generator=g, device="cuda", dtype=torch.uint8).view(torch.int8)
        m.input_factor.data = torch.randn(K, generator=g, device="cuda").half()
        m.weight_scale.data = (0.1 * torch.randn(N, generator=g, device="cuda")).half()
        x = torch.randn(T, K, generator=g, device="cuda").half()
        key = f"{T},{K},{N}"
        out["y" + key] = m(x).cpu().numpy()
        m.layernorm = nn.Identity()
        u = m(x)
        out["u" + key] = u.cpu().numpy()
        # (the same sums in 64 bits, and the bound: K / 32 float32 additions, two roundings to float16)
        a = (x * m.input_factor).double()
        s = 1.0 - 2.0 * ((m.weight.view(torch.uint8)[:, :, None] >> torch.arange(8, device="cuda", dtype=torch.uint8)) & 1).reshape(N, K).double()
        u64 = (a @ s.T) * m.weight_scale.double()
        bound = 2.01 * 2.0 ** -11 * u64.abs() + 4 * 2.0 ** -24 * K ** 0.5 * a.norm(dim=-1, keepdim=True) * m.weight_scale.double().abs() + 2.0 ** -24
        assert ((u.double() - u64).abs() <= bound).all(), (key, float(((u.double() - u64).abs() / bound).max()))
np.savez(sys.argv[1], **out)
"""


def _run(tmp, **env):
    path = os.path.join(str(tmp), "_".join(env.values()) + ".npz")
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", CHILD, path], cwd=root, env=dict(os.environ, **env), capture_output=True, text=True, timeout=110)
    assert r.returncode == 0, r.stdout + r.stderr
    return np.load(path)


@pytest.mark.parametrize("slices", ["0", "4"])
def test_every_tile_gives_the_same_product(tmp_path, slices):
    want = _run(tmp_path, OB_GEMM3_RT="8", OB_GEMM3_KSPLIT=slices)
    for rt in ("7", "6", "4", "3"):
        got = _run(tmp_path, OB_GEMM3_RT=rt, OB_GEMM3_KSPLIT=slices)
        for key in want.files:
            a, b = want[key].astype(np.float64), got[key].astype(np.float64)
            if slices == "0":
                assert np.array_equal(a, b), (rt, key)
            else:                                                            # (other tiles may take other slices: single roundings of u, y)
                assert np.linalg.norm(a - b) <= 1e-3 * np.linalg.norm(a), (rt, key)
