"""The text parser at the edges of its kernels: newlines at every offset of
the 16-byte loads and 64-byte masks, workgroups of 256 lines whose text fits
LDS (80 bytes per line) and just does not, empty and comment lines, chunks
that end inside a line, numbers of 1 to 40 digits.  The doubles are Python's
(correctly rounded), so they are compared for equality."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _parse(psh, tmp_path, text, n, fmtr, **kw):
    f = tmp_path / "c.txt"
    f.write_bytes(text)
    out = psh.DeviceArray.empty((max(n, 1), 4))
    ing = psh.Ingest(kw.pop("chunk", 0))
    ing.start_ascii(str(f), out, n, fmtr=fmtr, **kw)
    r = ing.wait()
    return r["n"], out.to_numpy((max(n, 1), 4))[:n]


@pytest.mark.parametrize("pad", [0, 1, 15, 16, 17, 42, 43, 63, 64, 65, 300])
@pytest.mark.parametrize("nlines,newline", [(1, True), (255, False), (256, True), (257, False),
                                            (1100, True)])
def test_line_offsets(psh, tmp_path, pad, nlines, newline):
    """Lines of 15 bytes and `pad` blanks (42: 57 bytes on average below the
    LDS limit, 65: 80 exactly, 300: above it), some empty or comments."""
    rng = np.random.default_rng(pad * 1000 + nlines)
    rows, lines = [], []
    for i in range(nlines):
        if i % 7 == 3:
            lines.append(["", "#" + "x" * (pad % 50), "  \t"][i // 7 % 3])
            continue
        v = rng.integers(0, 1000, 3)
        rows.append(v)
        lines.append(f"{v[0]:3d}.5 {v[1]:3d} {v[2]:4d}" + " " * pad)
    text = "\n".join(lines).encode() + (b"\n" if newline else b"")
    n, got = _parse(psh, tmp_path, text, len(rows), "%lf %lf %lf", comment="#")
    want = np.array(rows, float).reshape(-1, 3)
    want[:, 0] += 0.5
    assert n == len(rows) and np.array_equal(got[:, :3], want)


def test_number_lengths_and_chunks(psh, tmp_path):
    rng = np.random.default_rng(5)
    toks = []
    for k in range(3000):
        d = "".join(rng.choice(list("0123456789"), rng.integers(1, 41)))
        p = rng.integers(0, len(d) + 1)
        toks.append(("-" if k % 3 == 0 else "") + d[:p] + "." + d[p:] +
                    (f"e{rng.integers(-30, 30)}" if k % 4 == 0 else ""))
    text = "".join(f"{a} {b} {c}\n" for a, b, c in zip(toks[::3], toks[1::3], toks[2::3])).encode()
    want = np.array([float(t) for t in toks]).reshape(-1, 3)
    for chunk in (0, 37):      # 37 objects: chunks of 1776 bytes
        n, got = _parse(psh, tmp_path, text, 1000, "%lf %lf %lf", chunk=chunk)
        assert n == 1000 and np.array_equal(got[:, :3], want)
