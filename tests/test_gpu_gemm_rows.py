"""Linear layers of batches of prompts (csrc/gemm_rows.hip) at the edges of their tiles, in every form and with one to eight splits of the depth,
against products in 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DTYPES = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}      # half a unit in the last place of a result, relative


def _operands(M, N, K, dt, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(M, K + 8, generator=g, device="cuda").to(dt)[:, 8:]      # (rows further apart than they are long)
    w = torch.randn(N, K, generator=g, device="cuda").to(dt) * K ** -0.5
    z = x.double() @ w.double().t()
    # a float sum of K products in any order: each rounding is 2^-24 of a partial sum, none larger than the sum of magnitudes
    return x, w, z, K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())


# tiles of 64 to 192 rows and 64 to 256 columns: the last ones in part, one row and one column piece behind a tile, a slice of k and more than the slots hold; and deep
# products of few rows, whose depth is split
@pytest.mark.parametrize("M, N, K", [(65, 32, 64), (127, 96, 128), (129, 2048, 192), (200, 4096, 4096), (257, 2080, 512), (350, 4096, 2048), (512, 5120, 5120),
                                     (66, 2048, 5632), (96, 2080, 5632), (129, 4096, 11008), (193, 4128, 11008), (350, 2048, 5632), (700, 5120, 13824), (1024, 4096, 11008), (1000, 32, 4096)])
@pytest.mark.parametrize("dt", DTYPES)
def test_linear_rows(M, N, K, dt):
    from hydrainfer_amd._C.kernel.gemm import linear_rows
    x, w, z, eps = _operands(M, N, K, dt, M + N + K)
    got = linear_rows(x, w)
    assert got is not None and got.shape[-2:] == (M, N)
    if got.dim() == 3:
        assert got.dtype == torch.float32
        got = got.double().sum(dim=0)
    else:
        assert got.dtype == dt
        eps = eps + DTYPES[dt] * z.abs() + (2.0 ** -25 if dt == torch.float16 else 0)
    assert bool(((got.double() - z).abs() <= eps).all())


@pytest.mark.parametrize("M, N, K", [(65, 32, 64), (127, 96, 128), (129, 2080, 192), (104, 6144, 2048), (257, 4128, 512), (300, 6144, 2048), (1024, 4096, 2048), (1000, 32, 2048)])
@pytest.mark.parametrize("dt", DTYPES)
def test_linear_rows_whole(M, N, K, dt):
    from hydrainfer_amd._C.kernel.gemm import linear_rows_whole
    x, w, z, eps = _operands(M, N, K, dt, M + N + K)
    got = linear_rows_whole(x, w)
    assert got is not None and got.shape == (M, N) and got.dtype == dt
    assert bool(((got.double() - z).abs() <= eps + DTYPES[dt] * z.abs() + (2.0 ** -25 if dt == torch.float16 else 0)).all())


@pytest.mark.parametrize("M, N, K", [(64, 4096, 2048), (1025, 4096, 2048), (128, 2064, 2048), (128, 4096, 2080), (128, 6176, 2048), (128, 64, 4096)])
def test_linear_rows_whole_is_left_to_the_library(M, N, K):
    from hydrainfer_amd._C.kernel.gemm import linear_rows_whole
    x, w, _, _ = _operands(M, N, K, torch.bfloat16, 1)
    assert linear_rows_whole(x, w) is None


@pytest.mark.parametrize("M, N, K", [(64, 2048, 2048), (513, 2048, 2048), (1025, 2048, 5632), (128, 2064, 2048), (128, 2048, 2080)])
def test_linear_rows_is_left_to_the_library(M, N, K):
    from hydrainfer_amd._C.kernel.gemm import linear_rows
    x, w, _, _ = _operands(M, N, K, torch.bfloat16, 1)
    assert linear_rows(x, w) is None


@pytest.mark.parametrize("M, inter, K", [(65, 16, 128), (66, 5632, 2048), (129, 176, 192), (200, 11008, 4096), (317, 11008, 4096), (253, 13824, 5120), (600, 5632, 2048), (1024, 1040, 256)])
@pytest.mark.parametrize("dt", DTYPES)
def test_gate_up_of_fewer_rows(M, inter, K, dt):
    from hydrainfer_amd import _lib
    from hydrainfer_amd._C.kernel.gemm import gate_up_rows_supported, gate_up_silu_rows
    assert _lib.lib().hx_gate_up_silu_few_rows_supported(M, inter, K) == 1
    x, w, z, eps = _operands(M, 2 * inter, K, dt, M + inter)
    assert gate_up_rows_supported(x, w)
    got = gate_up_silu_rows(x, w).double()
    g, u = z[:, :inter], z[:, inter:]
    half = DTYPES[dt]
    dg, du = (eps[:, :inter] + half * g.abs() + 1e-7), (eps[:, inter:] + half * u.abs() + 1e-7)
    silu = g * torch.sigmoid(g)
    ds = 1.1 * dg + half * (silu.abs() + 1.1 * dg) + 1e-6      # |d silu / dg| < 1.1, rounded again
    want = silu * u
    bound = ds * (u.abs() + du) + silu.abs() * du
    assert bool(((got - want).abs() <= bound + half * (want.abs() + bound) + 1e-7).all())
