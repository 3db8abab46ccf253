"""The ears on the device (nunchi_amd.Ears, sh_ears_*) against the oracle restatement of imi's ears.

Every float table product, norm, conv, attention and the LayerNorm are the oracle's operations in the same order;
the device takes the double log10 of the mel sums and the erff of the projector's GELU from its own math library
where imi calls the C library, which may differ in the last place. So the mel frames and the rows are compared
within 1e-6 relative L2 (the oracle itself sits within 5e-5 of the float64 truth, tests/test_oracle_ears.py), and
the mel frames and rows before the first GELU difference are in practice equal bit for bit."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu
TOL = 1e-6


@pytest.fixture(scope="module")
def tiny_ears(model_dir):
    from nunchi_amd import synth
    return synth.cached("ears", synth.TINY_EARS, 3, model_dir)


@pytest.mark.parametrize("n", [1, 400, 401, 3 * 16000, 7 * 16000 + 123])
def test_tiny_ears_matches_oracle(tiny_ears, n):
    import nunchi_amd
    from nunchi_amd import synth
    pcm = synth.clip(n, 5)
    g = nunchi_amd.Ears(tiny_ears)
    out = g.encode(pcm)
    ref, mel = oracle.Ears(tiny_ears, threads=4).encode(pcm, mel=True)
    assert out.shape == ref.shape
    assert oracle.rel(g.mel(), mel) < TOL
    assert oracle.rel(out, ref) < TOL, oracle.rel(out, ref)


@pytest.mark.parametrize("n", [300, 5 * 16000 + 7])
def test_odd_table_sizes_match_oracle(model_dir, n):
    """Tables whose rows and columns end inside a 16-row tile and a 32-column chunk (8, 24, 40 and 264 columns, 264 rows)."""
    import nunchi_amd
    from nunchi_amd import synth
    shape = synth.EarsShape(n_mel=24, n_ch=8, n_embd=96, n_ff=40, n_head=3, n_head_kv=1, head_dim=32, layers="ca",
                            window=5, n_out=264)
    path = synth.cached("ears", shape, 4, model_dir)
    out = nunchi_amd.Ears(path).encode(synth.clip(n, 8))
    ref = oracle.Ears(path, threads=4).encode(synth.clip(n, 8))
    assert out.shape == ref.shape
    assert oracle.rel(out, ref) < TOL, oracle.rel(out, ref)


# rows and columns that end inside a table tile; the wide ones' clips give position tiles that a wave's 2 or 4 do not divide
SMALL = dict(n_mel=24, n_ch=8, n_embd=96, n_ff=40, n_head=3, n_head_kv=1, head_dim=32, layers="ca", window=5, n_out=264)
WIDE = dict(n_mel=128, n_ch=136, n_embd=96, n_ff=2056, n_head=32, n_head_kv=1, head_dim=128, layers="ca", window=5, n_out=264)
NORM = dict(n_mel=24, n_ch=8, n_ff=40, n_head=3, n_head_kv=1, head_dim=32, layers="c", window=5, n_out=264)


@pytest.mark.parametrize("kw,n", [(SMALL, 300), (SMALL, 5 * 16000 + 7), (WIDE, 384400)] +
                         [(dict(NORM, n_embd=E), 37123) for E in (256, 512, 768, 800)],
                         ids=["small-1", "small", "wide", "norm256", "norm512", "norm768", "norm800"])
def test_tables_bit_for_bit(model_dir, monkeypatch, kw, n):
    """The rows equal the oracle's bit for bit where erff cannot make a difference: with a projector bias of 50 every
    GELU input is far past the point from which erff is 1 in either library, so GELU is the identity in both."""
    import nunchi_amd
    from nunchi_amd import synth
    add = synth.GGUFWriter.add_tensor

    def biased(self, name, ty, dims, data):
        return add(self, name, ty, dims, np.full_like(data, 50.0) if name == "mm.a.mlp.1.bias" else data)
    monkeypatch.setattr(synth.GGUFWriter, "add_tensor", biased)
    path = synth.write_ears(f"{model_dir}/ears_bits_{kw['n_embd']}_{kw['n_ff']}.gguf", synth.EarsShape(**kw), 4)
    g = nunchi_amd.Ears(path)
    out = g.encode(synth.clip(n, 8))
    ref, mel = oracle.Ears(path, threads=8).encode(synth.clip(n, 8), mel=True)
    assert np.array_equal(g.mel().view(np.uint32), mel.view(np.uint32))
    assert out.shape == ref.shape
    assert np.array_equal(out.view(np.uint32), ref.view(np.uint32)), oracle.rel(out, ref)


def test_encode_repeats_and_shrinks(tiny_ears):
    """A longer clip, a shorter one (the work buffers are kept), then the first again: bit for bit the same rows."""
    import nunchi_amd
    from nunchi_amd import synth
    g = nunchi_amd.Ears(tiny_ears)
    a, b = synth.clip(5 * 16000, 6), synth.clip(16000, 7)
    ra = g.encode(a)
    rb = g.encode(b)
    assert np.array_equal(ra.view(np.uint32), g.encode(a).view(np.uint32))
    assert np.array_equal(rb.view(np.uint32), g.encode(b).view(np.uint32))


@pytest.mark.parametrize("n,rows", [(37123, 29), (384400, 301), (491760, 384)])
def test_full_ears(model_dir, n, rows):
    """The full ears shape on a short clip, on one whose position tiles leave a remainder in the waves of the pointwise and
    gate|up tables (1202 tiles by 4, 301 and 19 by 2), and on the 30.7 s of the hearing window."""
    import nunchi_amd
    from nunchi_amd import synth
    path = synth.cached("ears", synth.EARS, 3, model_dir)
    pcm = synth.clip(n, 1)
    out = nunchi_amd.Ears(path).encode(pcm)
    ref = oracle.Ears(path, threads=8).encode(pcm)
    assert out.shape == ref.shape == (rows, 2048)
    assert oracle.rel(out, ref) < TOL, oracle.rel(out, ref)


def test_bad_arguments_are_refused(tiny_ears):
    import nunchi_amd
    g = nunchi_amd.Ears(tiny_ears)
    with pytest.raises(nunchi_amd.SeoulError):
        g.encode(np.zeros(0, np.float32))


def test_mel_buffer_capacity_is_checked(tiny_ears):
    """sh_ears_mel writes only into a buffer that holds the last encode's frames: after a long clip, a buffer sized
    for a short one is refused with nothing written, and the binding sizes its buffer from the last encode."""
    import ctypes as C
    import nunchi_amd
    from nunchi_amd import synth
    g = nunchi_amd.Ears(tiny_ears)
    long_n, short_n = 7 * 16000 + 123, 16000
    g.encode(synth.clip(long_n, 5))
    _, f_long = g.positions(long_n)
    _, f_short = g.positions(short_n)
    assert f_short < f_long
    lib = nunchi_amd.load_library()
    buf = np.full((f_short + 1, g.info.n_mel), 7.0, np.float32)   # one guard frame past the capacity
    n = C.c_int(-1)
    rc = lib.sh_ears_mel(g.h, buf.ctypes.data, f_short, C.byref(n))
    assert rc == nunchi_amd.SH_E_ARG
    assert n.value == f_long
    assert np.all(buf == 7.0)
    m = g.mel()
    assert m.shape == (f_long, g.info.n_mel)
