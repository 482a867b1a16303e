"""The native binding (_native.so) without a GPU: one callable per declared
entry point with its argument count, and the torch operators' schemas."""

import pytest

from idempotent_llm_amd import _lib


def test_entries_cover_the_c_abi():
    entries = _lib.native().entries()
    assert set(entries) == set(_lib.SIGNATURES)
    for name, kinds in _lib.SIGNATURES.items():
        n = len(kinds) - (0 if name in _lib.HOST_ONLY else 1)
        with pytest.raises(TypeError, match=f"{name}: expected {n} arguments, got {n + 1}"):
            entries[name](0, *([0] * (n + 1)))


def test_argument_conversion_and_error_codes():
    """Empty problems return before any launch: ints, int-like objects, None
    and addresses convert; what does not convert raises; a negative return
    code raises with its value."""
    import numpy as np
    import torch
    t = torch.zeros(4, dtype=torch.int8)
    entries = _lib.native().entries()
    igemv = entries["detllm_igemv_nt"]
    for zero in (0, np.int64(0), torch.tensor(0), False):
        assert igemv(0, t, None, 0, zero, 16, 16, 1, 0) is None
    with pytest.raises(TypeError):
        igemv(0, t, None, 0, "0", 16, 16, 1, [])
    with pytest.raises(RuntimeError, match=r"detllm_igemv_nt failed \(code -22\)"):
        igemv(0, t, t, t, 65, 16, 16, 1, 0)
    with pytest.raises(RuntimeError, match=r"detllm_igemm_nt failed \(code -22\)"):
        _lib.native().entries()["detllm_igemm_nt"](0, t, t, t, 65, 16, 15, 1, 0, 0, 0)


def test_operators_mutate_what_they_declare():
    import torch

    from idempotent_llm_amd import torch_ops
    want = {"embed_normq": {"err"}, "residual_normq": {"h", "k_res"},
            "qkv_epilogue": {"kpool", "vpool", "err"}, "attn_decode": {"err"}}
    for name in torch_ops.OPS:
        op = getattr(torch.ops.detllm_rocm, name).default
        got = {a.name for a in op._schema.arguments if a.alias_info and a.alias_info.is_write}
        assert got == want.get(name, set()), name
        assert torch.Tag.pt2_compliant_tag in op.tags
        assert torch._C._dispatch_has_kernel_for_dispatch_key(f"detllm_rocm::{name}", "CUDA")
        assert not torch._C._dispatch_has_kernel_for_dispatch_key(f"detllm_rocm::{name}", "CPU")


# shapes int_gemm must refuse: a b of fewer or more rows than a's K (within
# and beyond the padded K), a batched b against one matrix, other batches
BAD_INT_GEMM = [((3, 16), (8, 5)), ((3, 16), (17, 5)), ((3, 100), (129, 5)), ((65, 200), (1, 40)),
                ((0, 16), (8, 5)), ((3, 16), (2, 16, 5)), ((4, 3, 16), (2, 16, 5)),
                ((2, 3, 3, 16), (3, 2, 16, 5)), ((4, 3, 16), (8, 5)), ((2, 3, 16), (2, 8, 5)),
                ((16,), (16, 5)), ((3, 16), (16,))]


@pytest.mark.parametrize("sa,sb", BAD_INT_GEMM)
def test_int_gemm_refuses_other_shapes(sa, sb):
    """The operator's kernels index b by a's shape, so operands that do not
    fit raise before any allocation or launch: called as the operator itself
    (the native kernel, on host tensors: no GPU work is reached) and traced."""
    import torch
    from torch._subclasses.fake_tensor import FakeTensorMode

    from idempotent_llm_amd import torch_ops  # noqa: F401
    op = torch.ops.detllm_rocm.int_gemm.default
    key = torch._C.DispatchKeySet(torch._C.DispatchKey.CUDA)
    a, b = torch.zeros(sa, dtype=torch.int8), torch.zeros(sb, dtype=torch.int8)
    with pytest.raises(ValueError):
        op.redispatch(key, a, b)
    with FakeTensorMode(), pytest.raises(ValueError):
        op(torch.empty(sa, dtype=torch.int8, device="cuda"),
           torch.empty(sb, dtype=torch.int8, device="cuda"))


def test_int_gemm_refuses_wide_elements():
    import torch

    from idempotent_llm_amd import torch_ops  # noqa: F401
    op = torch.ops.detllm_rocm.int_gemm.default
    key = torch._C.DispatchKeySet(torch._C.DispatchKey.CUDA)
    i8, i32 = torch.zeros(16, 16, dtype=torch.int8), torch.zeros(16, 16, dtype=torch.int32)
    for a, b in ((i8, i32), (i32, i8)):
        with pytest.raises(ValueError):
            op.redispatch(key, a, b)
