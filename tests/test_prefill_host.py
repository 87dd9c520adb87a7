"""Host side of the prefill call, without a GPU: the library is a stand-in that
records its arguments, and torch's operators are watched while the call runs."""
from __future__ import annotations

import contextlib

import numpy as np
import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode


class _Lib:
    """The prefill entry points of the library."""

    def __init__(self, n_split=1, ws_bytes=0):
        self.n_split, self.ws_bytes = n_split, ws_bytes

    def halo_prefill_splits(self, *a):
        self.splits_args = a
        return self.n_split

    def halo_prefill_workspace_size(self, *a):
        return self.ws_bytes if a[-1] > 1 else 0

    def halo_prefill_attn_split(self, *a):
        self.attn_args = a
        return 0


@pytest.fixture
def host(monkeypatch):
    """prefill_attention on CPU tensors over a _Lib."""
    from halo_amd import prefill as P
    from halo_amd.decode import DESC_DTYPE
    lib = _Lib()
    monkeypatch.setattr(P.nat, "lib", lambda: lib)
    monkeypatch.setattr(P.nat, "stream_ptr", lambda s=None: 0)
    monkeypatch.setattr(P, "pack_descs", lambda chunks, **kw: (np.zeros(len(chunks), DESC_DTYPE), []))
    monkeypatch.setattr(P, "_f32_direct", lambda q, chunks: True)
    return lib


def _chunk(dtype, T=32, *, B=1, H_kv=2, D=64, **kw):
    from halo_amd.decode import ChunkRef
    shape = (H_kv, T, D) if kw.get("batch", -1) >= 0 else (B, H_kv, T, D)
    t = torch.zeros(shape, dtype=dtype)
    return ChunkRef(t, t, kw.pop("start", 0), kw.pop("causal", True), **kw)


class _Writes(TorchDispatchMode):
    """Names of the operators that allocate or write while ``inside`` is not set."""

    def __init__(self, state):
        super().__init__()
        self.state, self.outside = state, []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        out = func(*args, **(kwargs or {}))
        name = func.overloadpacket.__name__
        if name in ("clone", "copy_", "_to_copy", "fill_") or "empty" in name:
            if not self.state["inside"]:
                self.outside.append(name)
        return out


@pytest.mark.parametrize("dtype,direct", [(torch.bfloat16, True), (torch.float32, True), (torch.float32, False)])
@pytest.mark.parametrize("q_form", ["aligned", "offset", "strided"])
def test_device_work_is_on_the_given_stream(host, monkeypatch, dtype, direct, q_form):
    """Copies of q, the output and the workspace belong to ``stream``: made
    elsewhere they would not be ordered with the kernels, and their memory
    could be handed out again while the kernels still use it."""
    from halo_amd import decode
    from halo_amd import prefill as P
    state = {"inside": False}

    @contextlib.contextmanager
    def on(stream):
        state["inside"] = True
        yield
        state["inside"] = False

    monkeypatch.setattr(torch.cuda, "stream", on)
    monkeypatch.setattr(P, "_f32_direct", lambda q, chunks: direct)
    monkeypatch.setattr(decode, "build_plan", lambda **kw: None)
    monkeypatch.setattr(decode, "launch", lambda *a, **kw: None)
    q = torch.zeros((1, 4, 8, 64), dtype=dtype)
    if q_form == "offset":
        q = torch.zeros(q.numel() + 1, dtype=dtype)[1:].view(q.shape)
    elif q_form == "strided":
        q = torch.zeros((1, 4, 8, 128), dtype=dtype)[..., ::2]
    with _Writes(state) as seen:
        P.prefill_attention(q, [_chunk(dtype)], return_lse=True, stream=object())
    assert seen.outside == []


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_split_workspace_is_bounded(dtype):
    """The library's choice of key splits takes at most 256 MiB of partials,
    whatever the rows and keys (2304 and 4100 rows are just past a round of
    workgroups in 16 and 32 bits), and does split where that is little."""
    from halo_amd import _native as nat
    if not nat.loadable():
        pytest.skip("library not built (run __graft_entry__.build())")
    L, dt = nat._load(), nat.dtype_code(dtype)
    split = 0
    for B in (1, 2, 4, 16):
        for H, H_kv, D in ((32, 8, 128), (28, 4, 128), (16, 4, 64), (8, 8, 64)):
            for T_q in (1, 137, 512, 1100, 2080, 2304, 4100, 4160, 8392, 33000):
                for prior in (0, 2048, 32768, 131072, 1 << 20):
                    s = L.halo_prefill_splits(dt, B, H, H_kv, T_q, D, prior + T_q, T_q)
                    assert L.halo_prefill_workspace_size(dt, B, H, H_kv, T_q, D, s) <= 256 << 20
                    split += s > 1
    assert split > 100


def test_call_without_memory_for_the_partials_runs_unsplit(host, monkeypatch):
    from halo_amd import prefill as P
    host.n_split, host.ws_bytes = 4, 1 << 20
    real = torch.empty

    def empty(*a, **kw):
        if kw.get("dtype") == torch.uint8:
            raise torch.OutOfMemoryError("no room")
        return real(*a, **kw)

    monkeypatch.setattr(torch, "empty", empty)
    P.prefill_attention(torch.zeros((1, 4, 8, 64), dtype=torch.bfloat16), [_chunk(torch.bfloat16)])
    assert host.attn_args[-4:-1] == (1, None, 0)
    monkeypatch.setattr(torch, "empty", real)
    P.prefill_attention(torch.zeros((1, 4, 8, 64), dtype=torch.bfloat16), [_chunk(torch.bfloat16)])
    assert host.attn_args[-4] == 4 and host.attn_args[-2] == 1 << 20


@pytest.mark.parametrize("batches,causal,want", [
    ((-1, -1, -1), (False, False, True), (96, 32)),   # every row reads every chunk
    ((0, 1, 2), (True, True, True), (32, 32)),        # one chunk a row
    ((0, 0, 2), (False, True, True), (64, 32)),       # the row with most keys
    ((-1, 1, 1), (False, False, True), (96, 32)),     # shared rows and a row's own
    ((-1, 0, -1), (False, True, True), (96, 64)),
])
def test_split_rule_gets_the_longest_walk(host, batches, causal, want):
    """The keys of one batch row and not those of the whole list: chunks of
    other rows are not part of a workgroup's walk."""
    from halo_amd import prefill as P
    chunks = [_chunk(torch.bfloat16, B=3, batch=b, causal=c) for b, c in zip(batches, causal)]
    P.prefill_attention(torch.zeros((3, 4, 8, 64), dtype=torch.bfloat16), chunks, q_start=0)
    assert host.splits_args[-2:] == want


@pytest.mark.parametrize("q_start", [torch.zeros(3, dtype=torch.int64), torch.zeros(0, dtype=torch.int64)])
@pytest.mark.parametrize("direct", [True, False])
def test_fp32_q_start_of_the_wrong_length(host, monkeypatch, q_start, direct):
    """Both fp32 forms refuse it by name."""
    from halo_amd import prefill as P
    monkeypatch.setattr(P, "_f32_direct", lambda q, chunks: direct)
    q = torch.zeros((2, 4, 8, 64))
    with pytest.raises(AssertionError, match="q_start must have B=2 entries"):
        P.prefill_attention(q, [_chunk(torch.float32, B=2)], q_start=q_start)


def test_fp32_chunks_without_a_batch():
    """The row form needs k, v, chunk_start and causal of a chunk and no more:
    an object with just these stays with it."""
    from types import SimpleNamespace

    from halo_amd.prefill import _f32_direct
    q = SimpleNamespace(is_cuda=True, shape=(1, 4, 8, 64))
    k = torch.zeros((1, 2, 32, 64))
    assert not _f32_direct(q, [SimpleNamespace(k=k, v=k, chunk_start=0, causal=True)])
