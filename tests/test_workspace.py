"""The buffers of a forward pass (model._Workspace): a buffer fits every
request, and none outlives the layers."""

import pytest
import torch

from idempotent_llm_amd import artifact as art


def test_buffer_fits_every_request():
    """A layer of another shape or type under the same name gets a buffer of
    its own (the kernels write through its address)."""
    from idempotent_llm_amd.model import _Workspace
    ws = _Workspace("cpu")
    a = ws.buf("P", (2, 3), torch.int32)
    assert ws.buf("P", (2, 3), torch.int32) is a
    for shape, dt in (((4, 3), torch.int32), ((3, 4), torch.int32), ((4, 3), torch.int64),
                      ((1, 4, 3), torch.int64)):
        b = ws.buf("P", shape, dt)
        assert b.shape == shape and b.dtype == dt and b is not a


@pytest.mark.gpu
def test_no_buffer_outlives_the_layers(tmp_path):
    """When the LM head starts, a prefill holds its residual, operand rows and
    scales (5 bytes per element and 4 words per row), not its layers'
    products and contexts."""
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from idempotent_llm_amd.model import IntQwen3, KVCache
    print("[no buffer outlives the layers]", flush=True)
    held = []

    class Probe(IntQwen3):
        def _lm_head(self, x8, xm, xk):
            held.append(torch.cuda.memory_allocated())
            return super()._lm_head(x8, xm, xk)

    d = str(tmp_path)
    art.make_artifact(d, art.MID, 5)
    m = Probe(d, backend="rocm")
    B, T = 3, 500
    ids = torch.randint(0, m.vocab, (B, T), device="cuda")
    pos = torch.arange(T, device="cuda").expand(B, T).contiguous()
    rows = torch.zeros(B, dtype=torch.int64, device="cuda")
    for _ in range(2):          # the first pass also makes what the model keeps
        cache = KVCache().plan(m, B, T)
        cache.reserve(m, B, T)
        before = torch.cuda.memory_allocated()
        m._forward(ids, pos, cache, None, rows)
    R, H = B * T, m.hidden
    assert held[-1] - before <= R * H * 5 + R * 8 * 4 + (1 << 20)
