"""Device-side loader conversion (src/nii2mesh.c:155-172) against the oracle,
bit for bit, for every datatype the CLI reads."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dtype,code', [(np.uint8, 2), (np.int16, 4), (np.uint16, 512), (np.float32, 16)])
@pytest.mark.parametrize('slope,inter', [(1.0, 0.0), (0.0, 0.0), (0.003921569, -0.5), (-2.75, 1000.125)])
def test_decode_matches_oracle(gpu, oracle, dtype, code, slope, inter):
    rng = np.random.default_rng(code)
    if dtype == np.float32:
        raw = rng.normal(0, 1000, (17, 19, 23)).astype(np.float32)
    else:
        info = np.iinfo(dtype)
        raw = rng.integers(info.min, info.max, (17, 19, 23), endpoint=True).astype(dtype)
    got = gpu.decode(raw, code, slope, inter)
    rc, want = oracle.decode(raw, code, slope, inter)
    assert rc == 0 and np.array_equal(got.ravel(), want)


def test_decode_rejects_other_types(gpu):
    with pytest.raises(RuntimeError):
        gpu.decode(np.zeros(8, np.int32), 8)


@pytest.mark.parametrize('dtype,code', [('uint8', 2), ('int16', 4), ('uint16', 512), ('float32', 16)])
@pytest.mark.parametrize('n', [1, 7, 8, 9, 4099])
@pytest.mark.parametrize('shift', [0, 1])
def test_decode_tails_and_alignment(gpu, dtype, code, n, shift):
    """Device decode of n voxels from and to arrays that start `shift`
    elements past an aligned address: whole packs, remainders, and the form
    without wide loads."""
    import ctypes as C
    import torch
    raw = np.arange(n + shift, dtype=np.int64) * 37 % 251
    raw = raw.astype(dtype)
    d = torch.from_numpy(raw.view(np.uint8).copy()).cuda()
    out = torch.full((n + shift + 8,), -1.0, dtype=torch.float32, device='cuda')
    torch.cuda.synchronize()
    with gpu.DeviceContext() as ctx:
        f = ctx.L.n2m_ctx_decode
        f.argtypes = [C.c_void_p, C.c_void_p, C.c_int, C.c_int64, C.c_float, C.c_float, C.c_void_p]
        assert f(ctx.h, d.data_ptr() + shift * raw.itemsize, code, n, 1.7, -3.3, out.data_ptr() + 4 * shift) == 0
    e = (raw[shift:].astype(np.float32) * np.float32(1.7)) + np.float32(-3.3)
    o = out.cpu().numpy()
    assert np.array_equal(o[shift:shift + n], e)
    assert (o[:shift] == -1).all() and (o[shift + n:] == -1).all()
