"""vmmul with its lines placed over the XCDs (8 lines and more, up to 64 MB) and
not: line counts around multiples of eight, lines that end at and beside a
workgroup, both dimensions, row- and column-major, real and complex operands, in
place, and a matrix on each side of the size rule.

Tolerance: a complex product is two roundings of each of its four terms: rel-L2
below 4 * 6e-8 = 2.4e-7."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("rows,cols", [(7, 300), (8, 1), (8, 256), (9, 257), (17, 255), (40, 513), (3000, 9), (8, 70000),
                                       (129, 65536), (127, 65536)])
@pytest.mark.parametrize("vtype,mtype", [("c", "c"), ("f", "c"), ("c", "f"), ("f", "f")])
def test_lines(ovx, rows, cols, vtype, mtype):
    import torch
    gen = torch.Generator(device="cuda").manual_seed(rows * 7 + cols)
    kind = {"c": torch.complex64, "f": torch.float32}
    m = torch.randn(rows, cols, dtype=kind[mtype], device="cuda", generator=gen)
    v0 = torch.randn(cols, dtype=kind[vtype], device="cuda", generator=gen)
    v1 = torch.randn(rows, dtype=kind[vtype], device="cuda", generator=gen)
    some = sorted({0, rows // 2, rows - 1})
    wide = {np.dtype("complex64"): np.complex128, np.dtype("float32"): np.float64}

    def up(t):
        a = t.cpu().numpy()
        return a.astype(wide[a.dtype])

    for dim, v in ((0, v0), (1, v1)):
        want = up(m[some]) * (up(v)[None, :] if dim == 0 else up(v)[some][:, None])
        got = ovx.vmmul(dim, v, m)
        assert rel(up(got[some]), want) < 2.4e-7
        if rows * cols < 1 << 20:
            t = m.t().contiguous().t()  # column-major
            out = torch.empty_like(got.t().contiguous()).t()
            ovx.vmmul(dim, v, t, out=out)
            assert torch.equal(out, got)
        if got.dtype == m.dtype:
            same = m.clone()
            ovx.vmmul(dim, v, same, out=same)
            assert torch.equal(same, got)
