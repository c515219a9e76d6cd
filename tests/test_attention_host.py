"""Host side of the attention call: which stream's memory its workspace is (kernels and tensors replaced, no GPU)."""
import contextlib
import types

import pytest
import torch


class _Lib:
    def xattn_block_sparse_workspace_bytes(self, *args):
        return 4096

    def xattn_block_sparse_fwd_ws(self, *args):
        self.args = args
        return 0


@pytest.mark.parametrize("side", [True, False])
def test_workspace_is_taken_on_the_stream_that_uses_it(monkeypatch, side):
    from xattn.src import Xattention as X

    lib, active, taken = _Lib(), ["current"], []

    @contextlib.contextmanager
    def on(stream):
        active.append(stream if stream is not None else active[-1])      # None: nothing changes
        yield
        active.pop()

    def empty(*size, **kw):
        t = make(*size, **kw)
        if kw.get("dtype") == torch.uint8:
            taken.append((active[-1], t.data_ptr()))
        return t

    make = torch.empty
    monkeypatch.setattr(X._hb, "lib", lambda: lib)
    monkeypatch.setattr(X, "_check_qk", lambda x, name: x)
    monkeypatch.setattr(X, "_stream_ptr", lambda dev: 1)
    monkeypatch.setattr(torch.cuda, "device", lambda dev: contextlib.nullcontext())
    monkeypatch.setattr(torch.cuda, "stream", on)
    monkeypatch.setattr(torch, "empty", empty)
    q = torch.zeros(1, 2, 256, 128, dtype=torch.bfloat16)
    stream = types.SimpleNamespace(cuda_stream=2) if side else None
    X.block_sparse_attention(q, q, q, stream=stream)
    assert taken == [(stream if side else "current", lib.args[4])]
    assert lib.args[-1] == (2 if side else 1)
