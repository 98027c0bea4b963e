"""The autotuner's choices saved to a text file and loaded into a fresh
context on the same lattice (ii_tune_save / ii_tune_load): the loaded
context writes the same file back, applies the network and the multi-rhs
hops without re-timing them, with results bitwise equal to the tuned
context's; a file for another lattice is refused."""
import numpy as np
import pytest

import iroiro_amd as ii
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def test_tune_file_round_trip(tmp_path):
    dims = (8, 8, 8, 16)
    lat = orc.Lattice(dims)
    u = lat.apbc(lat.gauge_expH(0.4, 91))
    b = np.random.default_rng(5).normal(size=(12, lat.half_size))
    outs = []
    files = [tmp_path / "a.tune", tmp_path / "b.tune"]
    for i in range(2):
        ctx = ii.Context(dims)
        try:
            ctx.upload_gauge(u)
            net = ii.LearnedPreconditioner(ctx)
            net.init_neumann(0.13, noise=0.3, seed=5)
            if i == 0:
                print(ctx.autotune())
                net.tune(12)
                ctx.tune_save(files[0])
            else:
                ctx.tune_load(files[0])
                ctx.tune_save(files[1])
            outs.append(net.apply_batched(b))
        finally:
            ctx.close()
    text = files[0].read_text()
    print(text)
    assert text == files[1].read_text()
    assert "hop " in text and "mrhs " in text and "net 12 " in text
    assert np.array_equal(outs[0], outs[1])
    other = ii.Context((8, 8, 8, 8))
    try:
        with pytest.raises(ii.IIError):
            other.tune_load(files[0])
    finally:
        other.close()


def hop_line(ctx, path):
    ctx.tune_save(path)
    return [v for v in path.read_text().splitlines() if v.startswith("hop ")]


def test_forced_hop_order_is_read_by_each_context(tmp_path, monkeypatch):
    """II_HOP_ORDER set after a context of the process has run its hops holds
    for the next context, and no longer once it is unset; the order changes no
    bit of the result."""
    dims = (16, 16, 4, 16)
    lat = orc.Lattice(dims)
    u = lat.apbc(lat.gauge_expH(0.4, 92))
    f = np.random.default_rng(6).normal(size=lat.half_size)
    res, lines = [], []
    for env in (None, "1:2", None):
        if env:
            monkeypatch.setenv("II_HOP_ORDER", env)
        else:
            monkeypatch.delenv("II_HOP_ORDER", raising=False)
        ctx = ii.Context(dims)
        res.append(ii.Dirac_Wilson_EvenOdd(0.1, u, ctx).mult(f))
        lines.append(hop_line(ctx, tmp_path / "t.tune"))
        ctx.close()
    assert lines[1][0].startswith("hop 1 2 ")
    assert not any(v.startswith("hop 1") for v in lines[0] + lines[2])
    assert np.array_equal(res[0], res[1]) and np.array_equal(res[0], res[2])


def test_file_of_an_untuned_context_leaves_the_hop_order(tmp_path, monkeypatch):
    """A context that has chosen no hop order writes none, and its file does not
    replace the order another context has."""
    dims = (16, 16, 4, 16)
    lat = orc.Lattice(dims)
    u = lat.apbc(lat.gauge_expH(0.4, 93))
    f = np.random.default_rng(7).normal(size=lat.half_size)
    plain, tuned = tmp_path / "plain.tune", tmp_path / "tuned.tune"
    monkeypatch.delenv("II_HOP_ORDER", raising=False)
    a = ii.Context(dims)
    ii.Dirac_Wilson_EvenOdd(0.1, u, a).mult(f)
    assert hop_line(a, plain) == []
    monkeypatch.setenv("II_HOP_ORDER", "1:2")
    b = ii.Context(dims)
    ii.Dirac_Wilson_EvenOdd(0.1, u, b).mult(f)
    want = hop_line(b, tuned)
    b.tune_load(plain)
    assert hop_line(b, tuned) == want and want[0].startswith("hop 1 2 ")
    a.close()
    b.close()


def test_multi_rhs_shapes_timed_where_blocks_are_few(tmp_path):
    """On a small lattice the tuner times every number of rhs per block: 64 tiles
    x 1 block of 12 rhs would leave most of the chip idle."""
    dims = (8, 8, 8, 16)
    ctx = ii.Context(dims)
    lat = orc.Lattice(dims)
    ctx.upload_gauge(lat.apbc(lat.gauge_expH(0.4, 94)))
    parts = ctx.autotune().split(";")
    mrhs = [p for p in parts if "multi-rhs hop" in p]
    assert len(mrhs) == 4
    for p in mrhs:
        for rb in (12, 6, 4, 3, 2):
            assert " %d/contig=" % rb in p
    ctx.close()


@pytest.mark.parametrize("line", ["mrhs 0 12 6 1 0 2 256", "mrhs 0 12 6 1 3 2 256",
                                  "mrhs 0 12 6 1 -1 2 256", "mrhs 0 12 6 7 2 2 256"])
def test_orders_the_lattice_does_not_have_are_contiguous(tmp_path, line):
    """An edited file's strip width that does not divide the time slices, or an
    unknown order, never reaches a kernel."""
    path = tmp_path / "t.tune"
    path.write_text("iroiro-hip tuning 1\nlattice 16 16 4 16\n" + line + "\n")
    ctx = ii.Context((16, 16, 4, 16))
    ctx.tune_load(path)
    ctx.tune_save(path)
    ctx.close()
    assert "mrhs 0 12 6 0 4 1 256" in path.read_text()
