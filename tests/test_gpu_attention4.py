"""The exact attention's kernels at the edges of their choice and of their
tiles, bit for bit against the CPU oracle.  The choice goes by the workgroups
that 16 and 32 query rows make (T rows, H heads), by T > 1024, and by what fits
in LDS (T <= 1344)."""
import pytest

import pyoracle as po
from pkgpu import Dev, bits_equal, describe_mismatch, pk

pytestmark = pytest.mark.gpu
SEED = 0x5EED4A00


@pytest.fixture(scope="module")
def dev():
    return Dev()


@pytest.mark.parametrize("T,H,pad", [
    # 16 rows a workgroup, staged: single rows, the edges of a tile of 16, the softmax's 8 and 64
    (1, 1, 0), (2, 3, 1), (15, 8, 0), (16, 8, 0), (17, 8, 3), (47, 2, 0), (65, 1, 1), (255, 2, 0), (512, 8, 0),
    # 32 rows, 8 waves
    (100, 40, 0), (33, 90, 2), (513, 8, 1),
    # 32 rows, 4 waves
    (101, 80, 0), (49, 150, 1), (31, 260, 0),
    # beyond T = 1024, the largest score rows in LDS, and the kernel past them
    (1025, 1, 0), (1344, 1, 1), (1345, 1, 0)])
def test_attention_kernels_bit_exact(dev, T, H, pad):
    D, lib = 128 * H, pk.load()
    ldq, ldp, ldo = 3 * D + 4 * pad, D + 4 * pad, D + pad
    qkv = po.normal((T, ldq), 0.0, 0.5, po.seed(SEED, f"q.{T}.{H}"))
    P = po.normal((2 * T - 1, ldp), 0.0, 0.5, po.seed(SEED, f"p.{T}.{H}"))
    pu, pv = (po.normal((D,), 0.0, 0.1, po.seed(SEED, f"{n}.{H}")) for n in "uv")
    dq, dP, du, dv = (dev.put(x) for x in (qkv, P, pu, pv))
    out = dev.torch.full((T, ldo), -7.0, device=dev.dev)
    n = lib.pk_gpu_attention_ws_floats(T, H)
    ws = dev.torch.empty(max(4, n), device=dev.dev)
    pk.call("pk_gpu_attention_ws_dev", dq.data_ptr(), ldq, dP.data_ptr(), ldp, du.data_ptr(), dv.data_ptr(),
            out.data_ptr(), ldo, T, H, ws.data_ptr(), n, dev.stream())
    got = out.cpu().numpy()
    assert (got[:, D:] == -7.0).all()                       # nothing written beside the rows
    want = po.attention_core(qkv[:, :3 * D].copy(), P[:, :D].copy(), pu, pv, H=H)
    got = got[:, :D].copy()
    assert bits_equal(got, want), describe_mismatch(got, want)
