"""The int8 products' kernels at the edges of their tile and dispatch rules,
against the product in float64 (sums of int8 products stay below 2^53, so it
is exact). Zero tolerance."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from idempotent_llm_amd import _lib
    _lib.load()


def _i8(seed, *shape):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randint(-128, 128, shape, dtype=torch.int8, device="cuda", generator=g)
    x.view(-1)[:4] = -128
    return x


def _want(a, bt):
    return (a.double() @ bt.double().t()).to(torch.int32)


@pytest.mark.parametrize("M", [1, 16, 17, 33, 49, 64])
@pytest.mark.parametrize("N,K", [(32768, 64), (32775, 1024), (33001, 1040), (32770, 4096)])
def test_head_product(M, N, K):
    """k_gemv_stream at each row-group count, ragged columns, K past one
    1024-byte step and K beyond what its LDS holds at M rows."""
    from idempotent_llm_amd.backends import gemm_nt
    print(f"[head product M={M} N={N} K={K}]", flush=True)
    a, w = _i8(M, M, K), _i8(N + K, N, K)
    out = torch.full((1, M, N), 7, dtype=torch.int32, device="cuda")
    gemm_nt(a, w, out=out)
    assert torch.equal(out[0], _want(a, w))
