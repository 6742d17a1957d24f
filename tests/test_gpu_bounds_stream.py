"""Block bounds of keys past the streaming size: the same values as torch's, NaN
and infinities included, at a block size that is no multiple of the rows in
flight and with and without 16-bit bounds."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hkv,n,b,d,dtype,inside", [
    (3, 4099, 64, 128, torch.bfloat16, True),    # 201 MB: just past it
    (2, 4001, 50, 256, torch.float16, True),     # 204 MB, a partial batch of rows
    (1, 6000, 33, 128, torch.bfloat16, False),   # below it
])
def test_bounds_match_torch(hkv, n, b, d, dtype, inside):
    from strict_topk import bounds
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    gen = torch.Generator(device="cuda").manual_seed(n)
    k = torch.randn((hkv, n, b, d), generator=gen, device="cuda", dtype=dtype)
    assert (k.numel() * 2 >= 192 << 20) == inside
    k[0, 1, 3, 5] = float("nan")
    k[-1, -1, -1, -1] = float("nan")
    k[0, 2, 0, 0], k[0, 2, 1, 0] = float("inf"), float("-inf")
    k[0, 3, :, 1] = 0.0
    for dt in (torch.float32, dtype):
        lo, hi = bounds.block_bounds(k, dt)
        for x, y in ((lo, k.amin(2)), (hi, k.amax(2))):
            assert x.dtype == dt
            assert torch.equal(x.isnan(), y.isnan())
            x, y = x.float(), y.float()
            assert torch.equal(torch.where(x.isnan(), 7.0, x), torch.where(y.isnan(), 7.0, y))
