"""GPU tests of the prefill kernel's three-plane products: every fp32 K, V, Q and P value is
multiplied as three bf16 planes that together hold all its bits, or in fp32 where it is out of the
planes' range.  Sizes sit at the edges of the
tiles (32 keys, 32-query blocks, units of 4 slots, two key groups), values at the edges of the
planes' range."""
import numpy as np
import pytest

from tests.parity import ATTN_RTOL, rel_err

pytestmark = pytest.mark.gpu

D = 128


def _run(gpu, q, k, v, pos0, H, HKV, ws=None):
    import torch
    dev = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (q, k, v)]
    pos = torch.tensor([pos0], dtype=torch.int32, device="cuda")
    out = gpu.attn_prefill(dev[0], dev[1], dev[2], pos, gpu.AttnShape(H, HKV), ws=ws)
    torch.cuda.synchronize()
    return out.cpu().numpy()


def _exact(q, k, v, pos0, H, HKV, dtype=np.float64):
    B, G = q.shape[0], H // HKV
    qd, kd, vd = (x.astype(dtype) for x in (q.reshape(B, H, D), k, v))
    out = np.zeros((B, H, D), dtype)
    for b in range(B):
        T = pos0 + b + 1
        for h in range(H):
            s = kd[:T, h // G] @ qd[b, h] / np.sqrt(dtype(D))
            p = np.exp(s - s.max())
            out[b, h] = (p / p.sum()) @ vd[:T, h // G]
    return out


def _inputs(orc, B, pos0, H, HKV, seed):
    n = pos0 + B
    return (orc.normal((B, H * D), seed), orc.normal((n, HKV, D), seed + 1), orc.normal((n, HKV, D), seed + 2))


def _close(got, exact):
    """Single elements within the attention bar, and the 2-norm within 1e-6.  An fp32 score of |s| ~ 11
    over 48 roundings is off by ~1.2e-7 (times the softmax scale), the exponent's argument and the
    exponential by ~1e-7 each, the value sums by less: 2e-7 to 5e-7 together.  A second-order plane
    product left out (2^-18 of |q||k|) alone is 1.3e-6."""
    off = np.linalg.norm(got.astype(np.float64) - exact) / np.linalg.norm(exact)
    assert off <= 1e-6, off
    assert rel_err(got, exact) <= ATTN_RTOL


@pytest.mark.parametrize("H,HKV,B,pos0", [(4, 1, 1, 0), (4, 1, 31, 0), (4, 1, 33, 31), (8, 2, 32, 32), (8, 2, 65, 63),
                                          (8, 1, 40, 29), (5, 1, 97, 1), (2, 2, 129, 64), (6, 2, 64, 95),
                                          (4, 1, 16, 1000)])
def test_prefill_error_against_float64(orc, gpu, H, HKV, B, pos0):
    q, k, v = _inputs(orc, B, pos0, H, HKV, 31000 + B + pos0)
    exact = _exact(q, k, v, pos0, H, HKV)
    for ws in (None, gpu.PrefillWorkspace(B, H, HKV, max(pos0 + B, 4096))):
        got = _run(gpu, q, k, v, pos0, H, HKV, ws)
        _close(got, exact)


def test_prefill_small_and_large_magnitudes(orc, gpu):
    """V near 1e-33, and K near 1e30 against q near 1e-30, which gives ordinary scores.  Same bound as
    above."""
    H, HKV, B, pos0 = 4, 1, 40, 50
    q, k, v = _inputs(orc, B, pos0, H, HKV, 32000)
    got = _run(gpu, q * np.float32(2.0 ** -100), k * np.float32(2.0 ** 100), v * np.float32(2.0 ** -110), pos0, H, HKV)
    exact = _exact(q, k, v, pos0, H, HKV)
    _close(got.astype(np.float64) * 2.0 ** 110, exact)


@pytest.mark.parametrize("split", [False, True])
def test_prefill_infinite_and_huge_values(orc, gpu, split):
    """An infinite K element whose scores are -inf drops the key and leaves finite rows; a V element
    past bf16's largest value stays the finite number it is; an infinite V element gives an infinite
    output in its own column only; a NaN in V stays in its column."""
    H, HKV, B, pos0 = 4, 1, 70, 60
    q, k, v = _inputs(orc, B, pos0, H, HKV, 33000)
    ws = gpu.PrefillWorkspace(B, H, HKV, 4096) if split else None
    q[:, ::D] = np.abs(q[:, ::D]) + np.float32(0.1)  # element 0 of every head positive
    k[37, 0, 0] = -np.inf
    ref = _exact(q, k, v, pos0, H, HKV)
    assert np.isfinite(ref).all()
    _close(_run(gpu, q, k, v, pos0, H, HKV, ws), ref)
    v[5, 0, 9] = np.float32(3.4e38)
    v[11, 0, 17] = np.inf
    v[12, 0, 21] = np.nan
    with np.errstate(invalid="ignore"):
        ref = _exact(q, k, v, pos0, H, HKV)
    got = _run(gpu, q, k, v, pos0, H, HKV, ws)
    assert np.isposinf(got[..., 17]).all() and np.isnan(got[..., 21]).all()
    cols = [c for c in range(D) if c not in (9, 17, 21)]
    _close(got[..., cols], ref[..., cols])
    assert np.max(np.abs(got[..., 9] / ref[..., 9] - 1.0)) <= 1e-5  # one term rules the column: p's own error


@pytest.mark.parametrize("H,HKV,B,pos0", [(32, 8, 16, 100), (16, 8, 64, 40), (8, 1, 33, 0), (40, 8, 100, 20), (4, 1, 2, 61)])
def test_prefill_small_chunk_plans(orc, gpu, H, HKV, B, pos0):
    """Small chunks whose plan of at least four tiles a share does not split: the queried workspace
    gives them finer shares (some hold one tile or none), and a call without a workspace is still
    taken, unsplit.  Both against float64."""
    from exactinfer_amd import _capi
    import torch
    q, k, v = _inputs(orc, B, pos0, H, HKV, 34000 + B)
    exact = _exact(q, k, v, pos0, H, HKV)
    n = pos0 + B
    ws = gpu.PrefillWorkspace(B, H, HKV, n)
    assert ws.nbytes > 0
    _close(_run(gpu, q, k, v, pos0, H, HKV, ws), exact)
    dev = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (q, k, v)]
    pos = torch.tensor([pos0], dtype=torch.int32, device="cuda")
    out = torch.full((B, H, D), float("nan"), dtype=torch.float32, device="cuda")
    _capi.call("ei_attn_prefill_split", gpu._stream(), dev[0].data_ptr(), H * D, out.data_ptr(), dev[1].data_ptr(),
               dev[2].data_ptr(), pos.data_ptr(), B, H, HKV, D, gpu.default_scale(), n, None, 0)
    torch.cuda.synchronize()
    _close(out.cpu().numpy(), exact)


def _aligned256(n):
    return (n + 255) & ~255


def _layer(orc, gpu, kernel, H, HKV, B, pos0, seed, qs=1.0, ks=1.0, vs=1.0, edit=None):
    """One chunk through one of the three prefill kernels: "plain" (rows normed beforehand), "step"
    (q normed in the attention kernel) or "paged" (32-row blocks in reversed order).  qs and ks scale
    the norms' gammas (and the past keys), vs all values; edit(k, v, qkv) changes the past rows and the
    raw chunk.  Returns the output and the operands q, k, v it was computed from."""
    import torch
    n, kd = pos0 + B, HKV * D
    qkv = orc.normal((B, (H + 2 * HKV) * D), seed)
    k, v = orc.normal((n, HKV, D), seed + 1) * np.float32(ks), orc.normal((n, HKV, D), seed + 2) * np.float32(vs)
    qkv[:, (H + HKV) * D:] *= np.float32(vs)
    qg, kg = orc.gamma(D, seed + 3) * np.float32(qs), orc.gamma(D, seed + 4) * np.float32(ks)
    if edit:
        edit(k, v, qkv)
    normed = orc.headnorm_rope(qkv, H, D, qg, pos0, 128, 1e6, 1e-6)
    normed = orc.headnorm_rope(normed, HKV, D, kg, pos0, 128, 1e6, 1e-6, col0=H * D)
    q = np.ascontiguousarray(normed[:, :H * D])
    k[pos0:] = normed[:, H * D:(H + HKV) * D].reshape(B, HKV, D)
    v[pos0:] = normed[:, (H + HKV) * D:].reshape(B, HKV, D)
    shape = gpu.AttnShape(H, HKV)
    ws = gpu.PrefillWorkspace(B, H, HKV, n)
    if kernel == "plain":
        return _run(gpu, q, k, v, pos0, H, HKV, ws), q, k, v
    past_k, past_v = k.copy(), v.copy()
    past_k[pos0:], past_v[pos0:] = 0, 0
    kw = {}
    if kernel == "paged":
        nblk = (n + 31) // 32
        table = np.arange(nblk - 1, -1, -1, dtype=np.int32)
        rows = table[np.arange(n) // 32] * 32 + np.arange(n) % 32
        pool = np.zeros((2, nblk * 32, HKV, D), np.float32)
        pool[0, rows], pool[1, rows] = past_k, past_v
        past_k, past_v = pool
        kw = dict(block_table=torch.from_numpy(table).cuda(), block_size=32)
    dev = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (qkv, past_k, past_v, qg, kg)]
    pos = torch.tensor([pos0], dtype=torch.int32, device="cuda")
    out = gpu.prefill_step(dev[0], dev[1].view(-1, kd), dev[2].view(-1, kd), shape, dev[3], dev[4], gpu.rope_table(n),
                           pos, ws, **kw)
    torch.cuda.synchronize()
    return out.cpu().numpy(), q, k, v


KERNELS = ["plain", "step", "paged"]


@pytest.mark.parametrize("kernel", KERNELS)
@pytest.mark.parametrize("e", [-112, -118, -124])
def test_prefill_tiny_values(orc, gpu, kernel, e):
    """V too small for three bf16 planes (whose smallest step is 2^-133), everywhere and in one column of
    ordinary values, and a column of zeros.  Same bound as above, column by column: the smallest outputs are
    fp32 denormals, whose step of 2^-149 is 2^-22 of them."""
    H, HKV, B, pos0 = 4, 1, 40, 50
    got, q, k, v = _layer(orc, gpu, kernel, H, HKV, B, pos0, 35000 - e, vs=2.0 ** e)
    _close(got.astype(np.float64) * 2.0 ** -e, _exact(q, k, v, pos0, H, HKV) * 2.0 ** -e)

    def columns(_, pv, qkv):
        chunk = qkv[:, (H + HKV) * D:]
        pv[..., 7] *= np.float32(2.0 ** e)
        chunk[:, 7] *= np.float32(2.0 ** e)
        pv[..., 77], chunk[:, 77] = 0, 0
    got, q, k, v = _layer(orc, gpu, kernel, H, HKV, B, pos0, 35100 - e, edit=columns)
    exact = _exact(q, k, v, pos0, H, HKV)
    _close(np.delete(got, 7, axis=-1), np.delete(exact, 7, axis=-1))
    assert (got[..., 77] == 0).all()
    _close(got[..., 7].astype(np.float64) * 2.0 ** -e, exact[..., 7] * 2.0 ** -e)


@pytest.mark.parametrize("kernel", KERNELS)
@pytest.mark.parametrize("e", [-120, 100, 120])
def test_prefill_q_out_of_plane_range(orc, gpu, kernel, e):
    """Tiny q against large K, and K too small for its planes against a q large enough to show it: ordinary
    scores, same bound."""
    H, HKV, B, pos0 = 8, 2, 40, 50
    got, q, k, v = _layer(orc, gpu, kernel, H, HKV, B, pos0, 36000 + e, qs=2.0 ** e, ks=2.0 ** -e)
    _close(got, _exact(q, k, v, pos0, H, HKV))


@pytest.mark.parametrize("split", [False, True])
def test_prefill_q_past_bf16_range(orc, gpu, split):
    """A finite q element above bf16's largest value, whose products with small K elements are ordinary."""
    H, HKV, B, pos0 = 4, 1, 40, 50
    q, k, v = _inputs(orc, B, pos0, H, HKV, 36500)
    q[:, 5::D] = np.float32(3.4e38)
    k[..., 5] *= np.float32(3e-39)
    got = _run(gpu, q, k, v, pos0, H, HKV, gpu.PrefillWorkspace(B, H, HKV, pos0 + B) if split else None)
    _close(got, _exact(q, k, v, pos0, H, HKV))


@pytest.mark.parametrize("split", [False, True])
def test_prefill_tiny_weights_of_huge_values(orc, gpu, split):
    """Keys of weight near 2^-122 that alone hold a column, with values that make it O(1): the probability
    keeps its 24 bits.  The scores are exact (one q element), so a weight is off by the exponent's argument:
    three roundings of about 122 (2^-18 each) times ln 2, 8e-6, and the exponential's own 1e-7."""
    H, HKV, B, pos0 = 4, 1, 40, 50
    q, k, v = _inputs(orc, B, pos0, H, HKV, 37000)
    q[:], k[:] = 0, 0
    q[:, ::D] = 8
    cols = list(range(3, 19, 2))
    v[..., cols] = 0
    for i, c in enumerate(cols):  # 8 * (120 .. 120.7) * log2(e) / sqrt(128) = 122.4 .. 123.1
        k[3 * i, 0, 0] = np.float32(-(120.0 + 0.1 * i))
        v[3 * i, 0, c] = np.float32(2.0 ** 124 * (1 + 0.1 * i))
    got = _run(gpu, q, k, v, pos0, H, HKV, gpu.PrefillWorkspace(B, H, HKV, pos0 + B) if split else None)
    exact = _exact(q, k, v, pos0, H, HKV)
    rest = np.delete(np.arange(D), cols)
    _close(got[..., rest], exact[..., rest])
    assert np.max(np.abs(got[..., cols] / exact[..., cols] - 1.0)) <= 1e-5


@pytest.mark.parametrize("kernel", KERNELS)
def test_prefill_infinities_by_kernel(orc, gpu, kernel):
    """Infinite, NaN and huge V elements through each kernel: each stays in its own column."""
    def edit(_, v, __):
        v[5, 0, 9] = np.float32(3.4e38)
        v[11, 0, 17] = np.inf
        v[12, 0, 21] = np.nan
    for H, HKV in ((4, 1), (5, 1)):
        got, q, k, v = _layer(orc, gpu, kernel, H, HKV, 70, 60, 38000 + H, edit=edit)
        with np.errstate(invalid="ignore"):
            ref = _exact(q, k, v, 60, H, HKV)
        assert np.isposinf(got[..., 17]).all() and np.isnan(got[..., 21]).all()
        cols = np.delete(np.arange(D), (9, 17, 21))
        _close(got[..., cols], ref[..., cols])
        assert np.max(np.abs(got[..., 9] / ref[..., 9] - 1.0)) <= 1e-5


@pytest.mark.parametrize("B", [2, 33])
def test_prefill_nan_key_alone_in_its_share(orc, gpu, B):
    """A NaN key that is the only visible one of its share (one-tile shares, the first query at a tile's
    first key) makes the row NaN as it does unsplit; rows that do not see it stay finite."""
    H, HKV, pos0 = 4, 1, 224
    q, k, v = _inputs(orc, B, pos0, H, HKV, 39000)
    for t in (pos0, pos0 + 1):
        kn = k.copy()
        kn[t, 0, 3] = np.nan
        plain = _run(gpu, q, kn, v, pos0, H, HKV)
        split = _run(gpu, q, kn, v, pos0, H, HKV, gpu.PrefillWorkspace(B, H, HKV, pos0 + B))
        want = np.broadcast_to((np.arange(B) >= t - pos0)[:, None, None], plain.shape)
        assert (np.isnan(plain) == want).all() and (np.isnan(split) == want).all()


def test_prefill_workspace_of_the_coarser_plan(orc, gpu):
    """A workspace that holds the plan of at least four tiles a share (two shares here) and not the finer
    one is taken, used within its bytes, and refused when one byte short."""
    import torch
    from exactinfer_amd import _capi
    H, HKV, B, pos0 = 32, 8, 64, 300
    n, shape = pos0 + B, gpu.AttnShape(32, 8)
    need = _aligned256(2 * B * H * D * 4) + _aligned256(2 * B * H * 2 * 4)
    assert need < gpu.PrefillWorkspace(B, H, HKV, n).nbytes
    buf = torch.full((need + 4096,), 0x5A, dtype=torch.uint8, device="cuda")
    _, q, k, v = _layer(orc, gpu, "plain", H, HKV, B, pos0, 40000)
    qkv = orc.normal((B, (H + 2 * HKV) * D), 40000)
    qg, kg = orc.gamma(D, 40003), orc.gamma(D, 40004)
    exact = _exact(q, k, v, pos0, H, HKV)
    pos = torch.tensor([pos0], dtype=torch.int32, device="cuda")
    cs = gpu.rope_table(n)

    def call(step, nbytes):
        dev = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (qkv if step else q, k, v, qg, kg)]
        out = torch.full((B, H, D), float("nan"), dtype=torch.float32, device="cuda")
        head = (gpu._stream(), dev[0].data_ptr(), dev[0].stride(0), out.data_ptr(), dev[1].data_ptr(),
                dev[2].data_ptr(), pos.data_ptr(), B, H, HKV, D)
        tail = (gpu.default_scale(), n, buf.data_ptr(), nbytes)
        if step:
            _capi.call("ei_prefill_step", *head, dev[3].data_ptr(), dev[4].data_ptr(), cs.data_ptr(), shape.rope_dim,
                       float(shape.eps), *tail)
        else:
            _capi.call("ei_attn_prefill_split", *head, *tail)
        torch.cuda.synchronize()
        return out.cpu().numpy()

    for step in (False, True):
        _close(call(step, need), exact)
        assert bool((buf[need:] == 0x5A).all())
        with pytest.raises(Exception, match="workspace"):
            call(step, need - 1)
