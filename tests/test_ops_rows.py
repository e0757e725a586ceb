"""The row views that ops.swiglu hands its kernel (CPU: no kernel runs)."""
import pytest
import torch

from fastllm_py.kernels.ops import _rows


def _forms():
    b = torch.arange(4096, dtype=torch.float32).to(torch.float16)
    m = b[:768].view(8, 96)
    return {
        "contiguous": m, "left half": m[:, :48], "right half": m[:, 48:], "odd columns": m[:, 5:38],
        "every other row": m[::2, :40], "one row": m[3:4, 7:20], "one strided row": m[2:3, ::2],
        "vector": m[1], "strided vector": m[:, 3], "three dims": b[:960].view(4, 5, 48)[:, :, :20],
        "three dims, outer gap": b[:960].view(4, 5, 48)[::2], "not one row stride": b[:960].view(4, 5, 48)[:, :3, :20],
        "expanded rows": m[:1].expand(6, 96), "expanded columns": m[:, :1].expand(8, 16), "transposed": m.t(),
        "overlapping rows": b.as_strided((6, 10), (4, 1)), "column stride 2": m[:, ::2],
        "one column": m[:, 4:5], "one column, one row": m[2:3, 4:5],
    }


@pytest.mark.parametrize("name", list(_forms()))
def test_rows_keep_the_values(name):
    v = _forms()[name]
    cols = v.shape[-1]
    r = _rows(v, cols, torch.empty(v.shape, dtype=v.dtype))
    assert r.shape == (v.numel() // cols, cols) and torch.equal(r, v.reshape(-1, cols))
    assert r.stride(1) == 1 or cols == 1
    assert r.stride(0) >= cols


def test_halves_are_not_copied():
    m = torch.zeros(8, 96, dtype=torch.float16)
    out = torch.empty(8, 48, dtype=torch.float16)
    for half in (m[:, :48], m[:, 48:]):
        r = _rows(half, 48, out)
        assert r.data_ptr() == half.data_ptr() and r.stride() == (96, 1)


def test_shared_memory_with_out_is_copied():
    m = torch.arange(768, dtype=torch.float32).to(torch.float16).view(8, 96)
    for out in (m.view(-1)[:384].view(8, 48), m.view(-1)[384:].view(8, 48)):
        r = _rows(m[:, :48], 48, out)
        assert r.is_contiguous() and r.data_ptr() != m.data_ptr() and torch.equal(r, m[:, :48])
    whole = _rows(m, 96, m)  # the same rows in place stay in place
    assert whole.data_ptr() == m.data_ptr()
