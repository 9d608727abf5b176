"""GPU tests of the projection at the edges of its row layout: a launch gives every workgroup
ceil(n_out / 256) output rows, spread over its row groups and taken a few at a time, so the output
counts here leave workgroups, groups and batches partly filled (one output in all, one more than
fills 256 workgroups, one row short of whole batches), for 1 to 4 activation rows and each weight
type.  Bound as in test_gpu_project: 1e-5 of sum_i |w_i h_i| (float64)."""
import numpy as np
import pytest

from tests.test_gpu_project import QTYPES, W_F16, W_F32, W_Q8_0, _host, _project, _qweights, _weights, _wf

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wtype", [W_F32, W_F16] + QTYPES)
@pytest.mark.parametrize("E,n_out,rows", [(1024, 1, 1), (1024, 257, 2), (1024, 2303, 4), (2048, 70, 3), (2048, 4095, 1),
                                         (2560, 9, 1), (2560, 700, 3), (2560, 1535, 2), (4096, 300, 2), (4096, 1025, 1),
                                         (4096, 1793, 4), (5120, 13, 4), (5120, 1025, 1), (5120, 515, 2)])
def test_projection_partly_filled_launches(orc, gpu, wtype, E, n_out, rows):
    x = orc.normal((rows, E), 8900 + E) * np.float32(3.0)
    gamma = orc.gamma(E, 8901)
    if wtype in QTYPES:
        w, wf = _qweights(orc, n_out, E, wtype, 8902 + n_out)
        wf = wf.astype(np.float64)
    else:
        w = _weights(orc, n_out, E, wtype, 8902 + n_out)
        wf = _wf(w, wtype)
    got = _host(_project(gpu, x, gamma, w, wtype, n_out)).astype(np.float64)
    for b in range(rows):
        h = orc.rmsnorm(x[b], gamma).astype(np.float64)
        assert np.max(np.abs(got[b] - wf @ h) / (np.abs(wf) @ np.abs(h))) <= 1e-5


@pytest.mark.parametrize("E,rows", [(8192, 1), (8192, 3), (10240, 1), (10240, 2)])
def test_projection_f16_wide_partly_filled(orc, gpu, E, rows):
    n_out = 777
    x = orc.normal((rows, E), 8950) * np.float32(3.0)
    gamma = orc.gamma(E, 8951)
    w = _weights(orc, n_out, E, W_F16, 8952)
    got = _host(_project(gpu, x, gamma, w, W_F16, n_out)).astype(np.float64)
    for b in range(rows):
        h = orc.rmsnorm(x[b], gamma).astype(np.float64)
        assert np.max(np.abs(got[b] - _wf(w, W_F16) @ h) / (np.abs(_wf(w, W_F16)) @ np.abs(h))) <= 1e-5


@pytest.mark.parametrize("rows", [2, 4])
def test_projection_strided_rows(orc, gpu, rows):
    """Activation and output rows wider than the product's: nothing beyond the outputs is written."""
    import torch
    from exactinfer_amd import _capi
    E, n_out, xs, os_ = 1024, 515, 1040, 530
    x = orc.normal((rows, xs), 8960)
    gamma = orc.gamma(E, 8961)
    w, wf = _qweights(orc, n_out, E, W_Q8_0, 8962)
    xd, gd, wd = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (x, gamma, w))
    out = torch.full((rows, os_), 7.0, dtype=torch.float32, device="cuda")
    _capi.call("ei_qkv_project", gpu._stream(), xd.data_ptr(), xs, rows, E, gd.data_ptr(), 1e-6, wd.data_ptr(), W_Q8_0,
               n_out, out.data_ptr(), os_)
    got = _host(out).astype(np.float64)
    assert (got[:, n_out:] == 7.0).all()
    for b in range(rows):
        h = orc.rmsnorm(x[b, :E], gamma).astype(np.float64)
        wd64 = wf.astype(np.float64)
        assert np.max(np.abs(got[b, :n_out] - wd64 @ h) / (np.abs(wd64) @ np.abs(h))) <= 1e-5
