"""The Python layer's device scratch: every call has its own, so that calls on several streams (or from several threads
on one) do not meet in one buffer."""
import gc
import weakref

import numpy as np
import pytest


def test_calls_do_not_share_a_workspace(nn, monkeypatch):
    """Two calls whose launches may overlap hold different memory, a larger request replaces nobody's, and nothing keeps
    a call's memory once the call has returned."""
    ops, torch = nn.ops, nn.ops.torch
    real = torch.empty
    monkeypatch.setattr(torch, "empty", lambda n, **kw: real(n, dtype=kw["dtype"]))
    a, na = ops._get_workspace(1 << 12)
    b, nb = ops._get_workspace(1 << 12)
    c, nc = ops._get_workspace(1 << 16)
    assert (na, nb, nc) == (1 << 12, 1 << 12, 1 << 16)
    spans = sorted((t.data_ptr(), t.data_ptr() + n) for t, n in ((a, na), (b, nb), (c, nc)))
    assert all(spans[i][1] <= spans[i + 1][0] for i in range(2))
    assert ops._get_workspace(0) == (None, 0)
    gone = weakref.ref(c)
    del c
    gc.collect()
    assert gone() is None


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["dropout", "shared bias"])
def test_gradients_on_two_streams(nn, kind):
    """Two different gradient calls whose workspaces hold data of the call (keep words, bias copies), launched in turn on
    two streams with no order between them: bit for bit what each gives alone."""
    import torch
    rng = np.random.default_rng(3)
    H, D, L, B = 8, 64, 512, 8
    D_ = nn.DeviceArray.from_numpy

    def call(seed):
        q, k, v, dy = (D_(rng.standard_normal((H * D, L, B)).astype(np.float32), "bf16") for _ in range(4))
        bias = D_(rng.standard_normal((L, L, H)).astype(np.float32), "bf16") if kind == "shared bias" else None
        fdrop = nn.Dropout(0.3, seed) if kind == "dropout" else nn.identity
        y, _ = nn.dot_product_attention(q, k, v, bias, nheads=H, return_weights=False, fdrop=fdrop, save_for_backward=True)

        def grad():
            return [g for g in nn.dot_product_attention_grad(dy, q, k, v, bias, y=y, nheads=H, fdrop=fdrop) if g is not None]
        return grad

    calls = [call(1), call(2)]
    alone = [[g.to_numpy() for g in c()] for c in calls]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    got = []
    for _ in range(6):
        for i, (c, s) in enumerate(zip(calls, streams)):
            with torch.cuda.stream(s):
                got.append((i, c()))
    torch.cuda.synchronize()
    for i, grads in got:
        for g, ref in zip(grads, alone[i]):
            assert np.array_equal(g.to_numpy(), ref)
