"""The host layer's routing on CPU tensors: its device check is lifted and a plain-torch op stands in
for the kernel, so each broadcast form can be compared with the op's definition (CPU only)."""
from __future__ import annotations

import types

import pytest
import torch

from autokernel_amd.kernels import host


def _rope_rows(y, x, cos, sin, rep_inner):
    """ak_rope's contract: row r of x [rows, D] uses row (r // rep_inner) % table_rows."""
    assert x.dim() == cos.dim() == sin.dim() == 2 and all(t.is_contiguous() for t in (x, y, cos, sin))
    row = (torch.arange(x.shape[0]) // rep_inner) % cos.shape[0]
    c, s = cos[row], sin[row]
    a, b = x[:, ::2], x[:, 1::2]
    y[:, ::2], y[:, 1::2] = a * c - b * s, a * s + b * c


ROPE_FORMS = [  # x shape, table shape
    ((6, 8), (6, 4)), ((6, 8), (1, 4)), ((6, 8), (4,)), ((8,), (4,)), ((1, 8), (1, 4)),
    ((2, 3, 6, 8), (6, 4)), ((2, 3, 6, 8), (1, 1, 6, 4)), ((2, 3, 6, 8), (1, 6, 4)),
    ((2, 6, 3, 8), (6, 1, 4)), ((2, 6, 3, 8), (1, 6, 1, 4)), ((2, 3, 6, 8), (3, 6, 4)),
    ((2, 3, 6, 8), (2, 3, 6, 4)), ((2, 3, 6, 8), (2, 1, 1, 4)), ((2, 3, 6, 8), (2, 1, 6, 4)),
    ((2, 1, 6, 8), (2, 3, 6, 4)), ((6, 8), (2, 6, 4)), ((6, 8), (1, 6, 4)), ((6, 8), (1, 1, 1, 4)),
    ((1, 8), (5, 4)), ((3, 1, 8), (1, 1, 4)), ((0, 8), (1, 4)), ((2, 6, 1, 8), (6, 1, 4)),
    ((6, 6, 8), (6, 1, 4)), ((5, 2), (5, 1)),
]


@pytest.mark.parametrize("xs,cs", ROPE_FORMS)
@pytest.mark.parametrize("form", ["dense", "strided", "mixed dtypes", "sin broadcast"])
def test_rotary_embedding_table_forms(monkeypatch, xs, cs, form):
    """Every table shape that broadcasts against x[..., ::2] gives the definition's result (exact in
    float64) and its shape, for dense and strided operands and tables of different shapes."""
    monkeypatch.setattr(host, "_check", lambda *a: None)
    monkeypatch.setattr(host, "ops", types.SimpleNamespace(rope=_rope_rows))
    g = torch.Generator().manual_seed(len(xs) * 31 + len(cs))

    def rnd(*s, dtype=torch.float64):
        return torch.randint(-8, 9, s, generator=g).to(dtype)
    x, cos, sin = rnd(*xs), rnd(*cs), rnd(*cs)
    if form == "strided":
        x = rnd(*xs[:-1], xs[-1] + 4)[..., 2:-2]
        cos = rnd(*cs[::-1]).permute(*range(len(cs) - 1, -1, -1))
        sin = rnd(*cs[:-1], cs[-1] * 2)[..., ::2]
    elif form == "mixed dtypes":
        cos, sin = cos.to(torch.float32), sin.to(torch.float16)
    elif form == "sin broadcast":
        sin = rnd(cs[-1])
    want_dt = torch.float64
    a, b, c, s = x[..., ::2], x[..., 1::2], cos.to(want_dt), sin.to(want_dt)
    want = torch.stack((a * c - b * s, a * s + b * c), -1).flatten(-2)
    got = host.rotary_embedding(x, cos, sin)
    assert got.dtype == want_dt and got.shape == want.shape
    assert torch.equal(got, want)
