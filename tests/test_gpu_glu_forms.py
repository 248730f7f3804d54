"""GLU's 16-byte and single-element forms, bit for bit against the CPU oracle."""
import pytest

import pyoracle as po
from pkgpu import Dev, bits_equal, describe_mismatch, pk

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [1, 3, 4, 250, 1024, 1028])
@pytest.mark.parametrize("offset", [0, 1])              # floats past a 16-byte address
def test_glu_forms(D, offset):
    dev = Dev()
    for rows in (1, 5, 257):
        x = po.normal((rows, 2 * D), 0.0, 3.0, po.seed(0x5EED6100, f"glu.{rows}.{D}"))
        src = dev.torch.zeros(rows * 2 * D + 4, device=dev.dev)
        dst = dev.torch.full((rows * D + 8,), -7.0, device=dev.dev)
        src[offset:offset + rows * 2 * D] = dev.put(x).reshape(-1)
        pk.call("pk_gpu_glu_dev", src.data_ptr() + 4 * offset, dst.data_ptr() + 4 * offset, rows, D, dev.stream())
        got = dst.cpu().numpy()
        assert (got[:offset] == -7.0).all() and (got[offset + rows * D:] == -7.0).all()
        got, want = got[offset:offset + rows * D].reshape(rows, D), po.glu(x)
        assert bits_equal(got, want), f"{rows}: {describe_mismatch(got, want)}"
