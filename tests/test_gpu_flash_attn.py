"""flash_attn_bhwd (megaqwen/triton_flash_attn.py:27-171) on the GPU against the float64 oracle
(oracle/flash_attn_ref.py): every output within half an ulp of the output type of the exact
attention, plus FLASH_ATTN_ABS * max|v| (tests/tolerances.py); the argument contracts of
triton_flash_attn.py:38-50 on CUDA tensors."""
import numpy as np
import pytest
import torch

from oracle.flash_attn_ref import attention_bhwd
from tests.tolerances import FLASH_ATTN_ABS

pytestmark = pytest.mark.gpu


def _fa():
    from megaqwen_amd.flash_attn import flash_attn_bhwd
    return flash_attn_bhwd


def _inputs(shape, dtype, seed, mag=1.0):
    g = torch.Generator().manual_seed(seed)
    return [(torch.randn(shape, generator=g) * mag).to(dtype) for _ in range(3)]


def _half_ulp(x, dtype):
    mant, emin = (7, -126) if dtype == torch.bfloat16 else (10, -14)
    e = np.floor(np.log2(np.maximum(np.abs(x), 2.0 ** emin)))
    return 0.5 * 2.0 ** (e - mant)


def _check(out, q, k, v, scale=None):
    assert out.dtype == q.dtype and out.shape == q.shape
    ref = attention_bhwd(q.double().numpy(), k.double().numpy(), v.double().numpy(), scale)
    o = out.double().cpu().numpy()
    assert np.isfinite(o).all()
    err = np.abs(o - ref)
    bound = _half_ulp(np.maximum(np.abs(ref), np.abs(o)), q.dtype) + \
        FLASH_ATTN_ABS * float(v.double().abs().max())
    worst = np.unravel_index(np.argmax(err - bound), err.shape)
    assert (err <= bound).all(), (
        f"{int((err > bound).sum())} outputs out of bound; worst at {worst}: "
        f"got {o[worst]}, oracle {ref[worst]}, bound {bound[worst]}")
    return float(err.max())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("t", [1, 37, 1500])
def test_audio_tower_shapes(dtype, t):
    """B = 1, 14 heads of 64 (Qwen3-ASR-0.6B audio tower), default scale 1/8."""
    q, k, v = _inputs((1, 14, t, 64), dtype, seed=t)
    out = _fa()(q.cuda(), k.cuda(), v.cuda())
    torch.cuda.synchronize()
    _check(out.cpu(), q, k, v)


def test_batches_heads_scale_and_strided_inputs():
    """B = 2, H = 3, explicit scale, inputs that are [B, T, H, D] tensors viewed as [B, H, T, D]
    (non-contiguous: the front end makes them contiguous, as the reference does)."""
    g = torch.Generator().manual_seed(5)
    base = [torch.randn(2, 100, 3, 64, generator=g).to(torch.float16) for _ in range(3)]
    q, k, v = (x.transpose(1, 2) for x in base)
    out = _fa()(*(x.cuda() for x in (q, k, v)), scale=0.37)
    torch.cuda.synchronize()
    _check(out.cpu(), q.contiguous(), k.contiguous(), v.contiguous(), scale=0.37)


@pytest.mark.parametrize("scale", ["0.25", np.float32(0.25), torch.tensor(0.25)])
def test_scale_is_anything_float_takes(scale):
    """`scale` goes through float(): number-like objects and numeric strings alike."""
    q, k, v = (x.cuda() for x in _inputs((1, 2, 40, 64), torch.bfloat16, seed=6))
    assert torch.equal(_fa()(q, k, v, scale=scale), _fa()(q, k, v, scale=0.25))
    with pytest.raises(ValueError):
        _fa()(q, k, v, scale="a quarter")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_peaked_softmax(dtype):
    """Scores spanning hundreds (inputs of std 6): the running max moves often and most weights
    underflow; the online rescale must keep the result exact to the bound."""
    q, k, v = _inputs((1, 4, 700, 64), dtype, seed=11, mag=6.0)
    v = torch.randn(v.shape, generator=torch.Generator().manual_seed(12)).to(dtype)
    out = _fa()(q.cuda(), k.cuda(), v.cuda())
    torch.cuda.synchronize()
    _check(out.cpu(), q, k, v)


# (batch * heads, T): both query-block widths (32 queries per wave for the small grids, 64 once
# 32-query workgroups exceed one round of the chip) at the edges of a key tile, of a query block
# and of the four waves' ranges (waves without a tile, one tile each, uneven ranges)
@pytest.mark.parametrize("bh,t", [(3, 31), (3, 32), (3, 33), (2, 64), (2, 65), (3, 127), (2, 129),
                                  (1, 161), (400, 33), (400, 64), (220, 97), (160, 129),
                                  (130, 191)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("scale", [0.125, -0.2, 0.0])
def test_tile_edges(bh, t, dtype, scale):
    q, k, v = _inputs((1, bh, t, 64), dtype, seed=bh + t)
    out = _fa()(q.cuda(), k.cuda(), v.cuda(), scale=scale)
    torch.cuda.synchronize()
    _check(out.cpu(), q, k, v, scale)


# 64 queries per workgroup, 6 to 15 key tiles per wave: tiles copied two ahead are used, and T % 32
# != 0 leaves a partial last tile.  mag 6 with keys that grow along T: scores of later tiles exceed
# the softmax reference again and again, so that sums other than zero are rescaled
@pytest.mark.parametrize("bh,t", [(56, 781), (56, 1001), (14, 1801)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("scale,mag", [(0.125, 1.0), (-0.2, 1.0), (0.125, 6.0), (-0.125, 6.0)])
def test_wide_workgroups(bh, t, dtype, scale, mag):
    q, k, v = _inputs((1, bh, t, 64), torch.float32, seed=bh + t)
    if mag != 1.0:
        k = k * torch.linspace(0.2, 1.0, t)[:, None] * mag
        q = q * mag
    q, k, v = (x.to(dtype) for x in (q, k, v))
    out = _fa()(q.cuda(), k.cuda(), v.cuda(), scale=scale)
    torch.cuda.synchronize()
    _check(out.cpu(), q, k, v, scale)


def test_one_key():
    """T = 1: the weight is exactly 1, so the output is v (an infinite v gives no finite output:
    its dim meets the weight's lo part, 0)."""
    q, k, v = _inputs((1, 3, 1, 64), torch.bfloat16, seed=4)
    assert torch.equal(_fa()(q.cuda(), k.cuda(), v.cuda()).cpu(), v)
    v[0, 1, 0, 9] = float("inf")
    got = _fa()(q.cuda(), k.cuda(), v.cuda()).cpu()
    assert not torch.isfinite(got[0, 1, 0, 9])
    got[0, 1, 0, 9] = v[0, 1, 0, 9]
    assert torch.equal(got, v)


# 32 queries per workgroup, and 64
@pytest.mark.parametrize("bh,t", [(2, 70), (56, 1001)])
def test_unaligned_and_non_finite_inputs(bh, t):
    """Contiguous tensors that start 2 bytes into an allocation; an infinite value reaches only
    its own dim's outputs, a NaN query only its own row, and the rows past T of the last key tile
    (T % 32 != 0) add nothing."""
    q, k, v = _inputs((1, bh, t, 64), torch.bfloat16, seed=21)
    dev = []
    for x in (q, k, v):
        buf = torch.zeros(x.numel() + 1, dtype=x.dtype, device="cuda")
        buf[1:] = x.flatten().cuda()
        dev.append(buf[1:].view(x.shape))
    assert all(x.data_ptr() % 4 == 2 for x in dev)
    out = _fa()(*dev)
    torch.cuda.synchronize()
    _check(out.cpu(), q, k, v)
    want = out.cpu()
    v2, q2 = v.clone(), q.clone()
    v2[0, 0, t - 1, 5] = float("inf")
    q2[0, 1, 3, 7] = float("nan")
    got = _fa()(q2.cuda(), k.cuda(), v2.cuda()).cpu()
    # (NaN instead of inf where the weight is a power of two: its lo part is 0, and 0 * inf is NaN)
    assert not torch.isfinite(got[0, 0, :, 5]).any() and torch.isnan(got[0, 1, 3]).all()
    assert torch.isinf(got[0, 0, :, 5]).float().mean() > 0.5
    got[0, 0, :, 5] = want[0, 0, :, 5]
    got[0, 1, 3] = want[0, 1, 3]
    assert torch.equal(got, want)


def test_deterministic_and_stream_ordered():
    q, k, v = (x.cuda() for x in _inputs((1, 14, 333, 64), torch.bfloat16, seed=3))
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        a = _fa()(q, k, v)
        b = _fa()(q, k, v)
    s.synchronize()
    assert torch.equal(a, b)


def test_empty_and_argument_contracts():
    fa = _fa()
    z = torch.zeros(1, 14, 0, 64, dtype=torch.bfloat16, device="cuda")
    out = fa(z, z, z)
    assert out.shape == z.shape and out.dtype == z.dtype
    x = torch.zeros(1, 2, 4, 64, dtype=torch.bfloat16, device="cuda")
    with pytest.raises(ValueError, match="only supports fp16/bf16"):
        fa(x.float(), x.float(), x.float())
    with pytest.raises(ValueError, match=r"Expected q.ndim=4"):
        fa(x[0], x[0], x[0])
    with pytest.raises(ValueError, match="Shape mismatch"):
        fa(x, x[:, :, :3], x)
    y = torch.zeros(1, 2, 4, 128, dtype=torch.bfloat16, device="cuda")
    with pytest.raises(ValueError, match="Only head_dim=64 supported, got 128"):
        fa(y, y, y)
    with pytest.raises(ValueError, match="dtype"):
        fa(x, x.half(), x)
