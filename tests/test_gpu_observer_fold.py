"""GPU: the per-tensor observer's amax over every grid it launches: one value,
less than a workgroup, either side of the size up to which it runs two
workgroups per CU, and a tail of fewer than 8 elements.  Exact: a maximum."""

import pytest
import torch


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 255, 2056, 1 << 20, 8 * 256 * 8 * 256, 8 * 256 * 8 * 256 + 8, 5_000_003])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_per_tensor_amax(vqx, n, dtype):
    print(f"observer fold n={n} {dtype}", flush=True)
    fq = vqx.quantization.QuantizationSpec.from_str("int8,qs=per_tensor_symmetric,ahl=4").make_fake_quantize("cuda").cuda()
    g = torch.Generator(device="cuda").manual_seed(n)
    for step, at in enumerate((0, n // 2, n - 1)):
        x = torch.randn(n, generator=g, device="cuda").to(dtype)
        x[at] = -50.0 - step  # the maximum, by magnitude, in another workgroup each time
        fq(x)
        assert float(fq.amax_history.flatten()[0]) == 50.0 + step
    x[n // 3] = float("nan")
    fq(x)
    assert bool(fq.amax_history.flatten()[0].isnan())
