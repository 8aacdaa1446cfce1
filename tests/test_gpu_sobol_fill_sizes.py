"""nova_hip_sobol_fill around the size where it changes kernels: the samples of one call equal those
of calls of a few thousand samples each (the kernel the golden vectors pin), out-of-range
dimensions included."""
import pytest

gpu = pytest.mark.gpu


@gpu
@pytest.mark.parametrize("n", [(1 << 18) - 1, 1 << 18, (1 << 18) + 1, 1500007])
def test_large_calls_equal_small_calls(n):
    import torch
    from axomae_amd import nova_hip
    g = torch.Generator(device="cuda").manual_seed(n)
    idx = torch.randint(-(1 << 31), 1 << 31, (n,), device="cuda", generator=g).to(torch.int32)
    dims = torch.randint(0, 256, (n,), device="cuda", generator=g).to(torch.int32)
    dims[::1001] = 256
    dims[5::4099] = -1
    print(f"[sobol] {n} samples", flush=True)
    out, bits = nova_hip.sobol_fill(idx, dims, return_bits=True)
    parts = [nova_hip.sobol_fill(idx[k:k + 100003], dims[k:k + 100003], return_bits=True) for k in range(0, n, 100003)]
    assert torch.equal(bits, torch.cat([p[1] for p in parts]))
    assert torch.equal(out.view(torch.int32), torch.cat([p[0] for p in parts]).view(torch.int32))
    plain = nova_hip.sobol_fill(idx, dims)
    assert torch.equal(out.view(torch.int32), plain.view(torch.int32))
