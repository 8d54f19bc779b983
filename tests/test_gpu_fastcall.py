"""The native call path (cf_hip/_fastcall.cpp) against ops.py's own path: same
results, same errors, the caller's stream."""

from __future__ import annotations

import pytest
import torch

from cf_hip import layout as L
from cf_hip import ops
from kernels.paged_attention import chunked_prefill_attention, paged_attention


class _None:
    """A native path that takes no call."""

    def __getattr__(self, name):
        return lambda *a: None


def test_cpu_tensors_and_wrong_types_are_left_to_the_wrappers():
    fast = ops._fast()
    t = torch.zeros(2, 4, 64)
    for x in (t, None, 3, t.to("meta")):
        assert fast.paged_write(x, torch.zeros(2, dtype=torch.int64), torch.zeros(1, 16, 4, 64), None) is None
        assert fast.scale_quantize(x, None, False) is None
    with pytest.raises(TypeError):
        fast.paged_write(t)
    with pytest.raises(ValueError):
        ops.paged_write(t, torch.zeros(2, dtype=torch.int64), torch.zeros(1, 16, 4, 64))


def _inputs(gpu, dtype):
    g = torch.Generator(device=gpu).manual_seed(5)
    nb, h, d = 40, 2, 64
    k, v = (torch.randn(nb, 16, h, d, generator=g, device=gpu).to(torch.bfloat16) for _ in range(2))
    ks, vs = ops.fp8_amax_scale(k), ops.fp8_amax_scale(v)
    kc, vc = L.alloc_kv_cache(nb, 16, h, d, dtype, gpu, "paired")
    if dtype == torch.float8_e4m3fn:
        ops.fp8_quantize_kv(k, v, ks, vs, kc, vc)
    else:
        kc.copy_(k)
        vc.copy_(v)
        ks = vs = None
    q = torch.randn(3, 4, d, generator=g, device=gpu).to(torch.bfloat16)
    tables = torch.arange(36, dtype=torch.int32, device=gpu).view(3, 12)
    lens = torch.tensor([5, 100, 192], dtype=torch.int32, device=gpu)
    return k, v, kc, vc, ks, vs, q, tables, lens


def _calls(gpu, dtype):
    k, v, kc, vc, ks, vs, q, tables, lens = _inputs(gpu, dtype)
    start = torch.tensor([0, 1, 2, 3], dtype=torch.int32, device=gpu)
    slots = torch.tensor([7, -1, 300], dtype=torch.int64, device=gpu)
    rows = k[:3, 0]
    out = {
        "decode": ops.paged_decode(q, kc, vc, tables, lens, 0.125, 16, ks, vs),
        "shared": ops.paged_decode(q, kc, vc, tables, lens, 0.125, 16, ks, vs, shared_prefix_lens=lens * 0),
        "prefill": chunked_prefill_attention(q, kc, vc, tables, lens, start, k_scale=ks, v_scale=vs),
        "gather": ops.paged_gather(kc, tables, 50, scale=ks),
        "gather16": ops.paged_gather(kc, tables, 50, out_dtype=torch.float16, scale=ks),
        "dict": torch.stack(list(paged_attention(
            q, kc, vc, {f"r{i}": tables[i].tolist() for i in range(3)}, {"r0": 5, "r1": 100}, k_scale=ks,
            v_scale=vs).values())),
    }
    ops.paged_write(rows, slots, kc, ks)
    if ks is not None:
        ops.kv_write_fp8(rows, rows, slots + 400, kc, vc, ks, vs)
        out["codes"] = kc.view(torch.uint8)
    else:
        out["rows"] = kc
    return {name: t.clone() for name, t in out.items()}


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float8_e4m3fn])
def test_results_equal_the_wrappers_own_path(gpu, monkeypatch, dtype):
    got = _calls(gpu, dtype)
    side = torch.cuda.Stream(device=gpu)
    side.wait_stream(torch.cuda.current_stream(gpu))
    with torch.cuda.stream(side):  # the current stream is used, with a workspace of its own
        other = _calls(gpu, dtype)
    torch.cuda.synchronize()
    monkeypatch.setattr(ops, "_FAST", _None())
    want = _calls(gpu, dtype)
    for name in want:
        assert torch.equal(got[name], want[name]) and torch.equal(other[name], want[name]), name


@pytest.mark.gpu
def test_errors_are_the_wrappers(gpu, monkeypatch):
    k, v, kc, vc, ks, vs, q, tables, lens = _inputs(gpu, torch.bfloat16)
    bad = [
        lambda: ops.paged_decode(q, kc, vc, tables, lens.cpu(), 0.125, 16),
        lambda: ops.paged_decode(q, kc, vc, tables.long(), lens, 0.125, 16),
        lambda: ops.paged_decode(q, kc, vc, tables, lens, 0.125, 8),
        lambda: ops.paged_decode(q, kc, vc, tables, lens, 0.125, 16, partition_tokens=24),
        lambda: ops.paged_decode(q, kc, vc, tables, lens, 0.125, 16, out=q.float()),
        lambda: ops.paged_decode(q, kc, vc, tables, lens, 0.125, 16, workspace=q.new_empty(256)),
        lambda: ops.paged_decode(q.double(), kc, vc, tables, lens, 0.125, 16),
        lambda: ops.prefill_chunk(q, kc, vc, tables, lens, lens, 0.125),
        lambda: ops.prefill_chunk(q.float(), kc, vc, tables, lens, lens.new_zeros(4), 0.125),
        lambda: ops.paged_write(k[:3, 0], lens[:2], kc),
        lambda: ops.paged_write(k[:3, 0], lens, kc, scale=lens.float()),
        lambda: ops.paged_gather(kc, tables[0], 4),
        lambda: ops.kv_write_fp8(k[:3, 0], v[:3, 0], lens, kc, vc, lens.float(), lens.float()),
    ]

    def kinds():
        out = []
        for f in bad:
            with pytest.raises(Exception) as e:
                f()
            out.append((e.type, str(e.value)))
        return out

    got = kinds()
    monkeypatch.setattr(ops, "_FAST", _None())
    assert got == kinds()
