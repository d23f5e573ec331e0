"""Encoder-level parity on the GPU: the vision and text towers through the
C-ABI against the CPU oracle on identical seeded weights and inputs, plus
the batch / ragged invariances (a batched or packed image must produce the
same bits as that image alone)."""
import ctypes

import numpy as np
import pytest
import torch

import pyoracle
import s2x
from s2x import synth
from gemm_forms import F16_TOWER_ROWS
from gpu_util import cos, dev, empty, host, ptr, say

pytestmark = pytest.mark.gpu

SMALL_V = synth.VisionConfig(hidden=288, inter=1076, n_head=4, n_layer=2)
SMALL_T = synth.TextConfig(hidden=288, inter=1076, n_head=4, n_layer=2, vocab=1000, max_pos=64,
                           proj=288)


class Vision:
    def __init__(self, hostm):
        self.host = hostm
        self.h = ctypes.c_void_p()
        s2x.call("s2x_vision_create", ctypes.byref(hostm.struct), ctypes.byref(self.h))

    def encode(self, px, n_h, n_w, pooling):
        out = np.empty(self.host.cfg.hidden, np.float32)
        px = np.ascontiguousarray(px, np.float32)
        s2x.call("s2x_vision_encode", self.h, px.ctypes.data, n_h, n_w, pooling, out.ctypes.data)
        return out

    def batch(self, px, n_img, n_h, n_w, pooling):
        pd = dev(px)
        out = empty((n_img, self.host.cfg.hidden), torch.float32)
        s2x.call("s2x_vision_encode_batch_dev", self.h, ptr(pd), n_img, n_h, n_w, pooling, ptr(out))
        return host(out)

    def ragged(self, padded, shapes, max_patches, pooling):
        pd = dev(padded)
        sh = np.ascontiguousarray(shapes, np.int32)
        out = empty((len(shapes), self.host.cfg.hidden), torch.float32)
        s2x.call("s2x_vision_encode_ragged_dev", self.h, ptr(pd), sh.ctypes.data, len(shapes),
                 max_patches, pooling, ptr(out))
        return host(out)

    def close(self):
        s2x.lib.s2x_vision_destroy(self.h)


@pytest.fixture(scope="module")
def small_vision(orc):
    hm = synth.vision_model(SMALL_V, seed=21)
    v = Vision(hm)
    yield v, orc.vision_model(hm)
    v.close()


@pytest.mark.parametrize("grid", [(16, 16), (27, 27), (12, 20), (8, 32)])
@pytest.mark.parametrize("pooling", [s2x.POOL_PROBE, s2x.POOL_MEAN])
def test_small_vision_vs_oracle(orc, small_vision, grid, pooling):
    v, om = small_vision
    h, w = grid
    px = synth.pixels(1, h * w, seed=h * 31 + w)
    g = v.encode(px, h, w, pooling)
    r = orc.vision_encode(om, px, h, w, pooling=pooling)
    c = cos(g, r)
    say(f"small vision {grid} pooling={pooling}: cosine {c:.7f}")
    assert c >= 0.9999


def test_small_vision_batch_invariance(small_vision):
    v, _ = small_vision
    px = synth.pixels(3, 729, seed=5)
    b = v.batch(px, 3, 27, 27, s2x.POOL_PROBE)
    for i in range(3):
        one = v.batch(px[i * 729:(i + 1) * 729], 1, 27, 27, s2x.POOL_PROBE)
        assert np.array_equal(b[i], one[0]), i
    assert np.array_equal(v.encode(px[:729], 27, 27, s2x.POOL_PROBE), b[0])


@pytest.mark.parametrize("pooling", [s2x.POOL_PROBE, s2x.POOL_MEAN])
def test_small_vision_ragged_equals_per_image(small_vision, pooling):
    v, _ = small_vision
    shapes = [(16, 16), (12, 20), (27, 27), (24, 24), (32, 32)]
    maxp = 1024
    padded = np.zeros((len(shapes), maxp, 768), np.float32)
    singles = []
    for i, (h, w) in enumerate(shapes):
        px = synth.pixels(1, h * w, seed=100 + i)
        padded[i, :h * w] = px
        padded[i, h * w:] = 7.0  # padding content must not matter
        singles.append(v.batch(px, 1, h, w, pooling)[0])
    out = v.ragged(padded.reshape(-1, 768), shapes, maxp, pooling)
    for i in range(len(shapes)):
        assert np.array_equal(out[i], singles[i]), shapes[i]


@pytest.mark.parametrize("pooling", [s2x.POOL_PROBE, s2x.POOL_MEAN])
def test_small_vision_rgb_batch_equals_preprocessed(small_vision, pooling):
    # raw RGB images of assorted sizes through the GPU NaFlex front end and
    # the tower in one call == the oracle's preprocessing (the reference's
    # bits) fed to the ragged encode
    v, _ = small_vision
    sizes = [(480, 640), (300, 1000), (432, 432), (37, 53)]
    maxp, p = 576, 16
    rng = np.random.default_rng(91)
    imgs = [rng.integers(0, 256, (h, w, 3), dtype=np.uint8) for h, w in sizes]
    padded = np.zeros((len(sizes), maxp, 3 * p * p), np.float32)
    shapes = []
    for i, img in enumerate(imgs):
        pre, nh, nw = pyoracle.nf_preprocess_rgb(img, maxp, p=p, fused=1)
        padded[i, :nh * nw] = pre
        shapes.append((nh, nw))
    want = v.ragged(padded.reshape(-1, 3 * p * p), shapes, maxp, pooling)
    dimgs = [dev(np.ascontiguousarray(im)) for im in imgs]
    ptrs = (ctypes.c_void_p * len(imgs))(*[ptr(d) for d in dimgs])
    hw = np.array(sizes, np.int32)
    mean = np.array([0.5, 0.5, 0.5], np.float32)
    std = np.array([0.5, 0.5, 0.5], np.float32)
    out = empty((len(imgs), v.host.cfg.hidden), torch.float32)
    s2x.call("s2x_vision_encode_rgb_batch_dev", v.h, ptrs, hw.ctypes.data, len(imgs), maxp,
             ctypes.c_float(1.0 / 255.0), mean.ctypes.data, std.ctypes.data, pooling, ptr(out))
    assert np.array_equal(host(out), want)


def test_vision_rejects_bad_shapes(small_vision):
    v, _ = small_vision
    px = np.zeros((4, 768), np.float32)
    out = np.empty(288, np.float32)
    assert s2x.lib.s2x_vision_encode(v.h, px.ctypes.data, 0, 4, 1, out.ctypes.data) == 1
    sh = np.array([[40, 40]], np.int32)
    assert s2x.lib.s2x_vision_encode_ragged_dev(v.h, ctypes.c_void_p(1), sh.ctypes.data, 1, 1024, 1,
                                                ctypes.c_void_p(1)) == 1


class Text:
    def __init__(self, hostm):
        self.host = hostm
        self.h = ctypes.c_void_p()
        s2x.call("s2x_text_create", ctypes.byref(hostm.struct), ctypes.byref(self.h))

    def encode(self, ids, mask=None):
        out = np.empty(self.host.cfg.proj, np.float32)
        ids = np.ascontiguousarray(ids, np.int32)
        m = None if mask is None else np.ascontiguousarray(mask, np.int32)
        s2x.call("s2x_text_encode", self.h, ids.ctypes.data, ids.size,
                 None if m is None else m.ctypes.data, out.ctypes.data)
        return out

    def batch(self, ids):
        ids = np.ascontiguousarray(ids, np.int32)
        out = np.empty((ids.shape[0], self.host.cfg.proj), np.float32)
        s2x.call("s2x_text_encode_batch", self.h, ids.ctypes.data, ids.shape[1], ids.shape[0],
                 out.ctypes.data)
        return out

    def close(self):
        s2x.lib.s2x_text_destroy(self.h)


def test_vision_graph_replays_match_eager(small_vision):
    """Batch-size-1 encodes run as HIP graph replays from the second call
    with the same shape and buffers on.  Every call -- the first (plain
    launches), the capturing one and the replays, with another shape's
    encodes (cached as a second graph), op-level work on torch's stream and
    synchronisations between them -- gives the plain launches' bits."""
    v, _ = small_vision
    H = v.host.cfg.hidden
    a = dev(synth.pixels(1, 27 * 27, seed=6000))
    b = dev(synth.pixels(2, 16 * 16, seed=6001))
    oa, ob = empty((1, H), torch.float32), empty((2, H), torch.float32)

    def run_a():
        s2x.call("s2x_vision_encode_batch_dev", v.h, ptr(a), 1, 27, 27, s2x.POOL_PROBE, ptr(oa))
        return host(oa).copy()

    def run_b():
        s2x.call("s2x_vision_encode_batch_dev", v.h, ptr(b), 2, 16, 16, s2x.POOL_MEAN, ptr(ob))
        return host(ob).copy()

    s2x.call("s2x_vision_set_graphs", v.h, 0)
    try:
        ref_a, ref_b = run_a(), run_b()
    finally:
        s2x.call("s2x_vision_set_graphs", v.h, 1)
    scratch = empty((1 << 20,), torch.float32)
    for i in range(6):
        oa.fill_(float("nan"))
        ob.fill_(float("nan"))
        assert np.array_equal(run_a(), ref_a), f"27x27 call {i}"
        scratch.normal_()  # eager work on torch's stream between replays
        assert np.array_equal(run_b(), ref_b), f"2 x 16x16 call {i}"
        torch.cuda.synchronize()
    say("vision: 6 rounds of two shapes, graph replays equal plain launches")


def test_text_graph_replays_match_eager():
    hm = synth.text_model(SMALL_T, seed=23)
    t = Text(hm)
    try:
        rng = np.random.default_rng(24)
        ids = rng.integers(0, SMALL_T.vocab, (3, 20)).astype(np.int32)
        s2x.call("s2x_text_set_graphs", t.h, 0)
        ref = t.batch(ids)
        ref1 = t.encode(ids[0])
        s2x.call("s2x_text_set_graphs", t.h, 1)
        for i in range(5):
            assert np.array_equal(t.batch(ids), ref), f"batch call {i}"
            assert np.array_equal(t.encode(ids[0]), ref1), f"single call {i}"
    finally:
        t.close()


@pytest.mark.parametrize("fp64", [0, 1])
def test_small_text_vs_oracle(orc, fp64):
    # the flash (f16 MFMA) attention, the default, and the fp64 option
    hm = synth.text_model(SMALL_T, seed=22)
    t = Text(hm)
    try:
        s2x.call("s2x_text_set_attention_fp64", t.h, fp64)
        om = orc.text_model(hm)
        ids, lens = synth.text_tokens(5, 64, vocab=SMALL_T.vocab)
        b = t.batch(ids)
        for i in range(5):
            r = orc.text_encode(om, ids[i])
            assert cos(b[i], r) >= 0.9999
            assert np.array_equal(t.encode(ids[i]), b[i])
        mask = np.zeros(64, np.int32)
        mask[:lens[1]] = 1
        c = cos(t.encode(ids[1], mask), orc.text_encode(om, ids[1], mask))
        say(f"small text masked cosine {c:.7f}")
        assert c >= 0.9999
        short = ids[2, :17]
        assert cos(t.encode(short), orc.text_encode(om, short)) >= 0.9999
        bad = ids[0].copy()
        bad[3] = SMALL_T.vocab
        out = np.empty(SMALL_T.proj, np.float32)
        assert s2x.lib.s2x_text_encode(t.h, bad.ctypes.data, 64, None, out.ctypes.data) == 1
    finally:
        t.close()


# ---------------------------------------------------------------- so400m ----
@pytest.fixture(scope="module")
def so400m_vision(orc):
    say("generating so400m vision weights")
    hm = synth.vision_model(synth.SO400M_VISION, seed=0)
    v = Vision(hm)
    yield v, orc.vision_model(hm)
    v.close()


@pytest.mark.timeout(600)
def test_so400m_vision_729_probe_vs_oracle(orc, so400m_vision):
    v, om = so400m_vision
    px = synth.pixels(1, 729, seed=1234)
    g = v.encode(px, 27, 27, s2x.POOL_PROBE)
    say("oracle so400m tower (CPU)")
    r = orc.vision_encode(om, px, 27, 27, pooling=1)
    c = cos(g, r)
    say(f"so400m vision 27x27 probe: cosine {c:.7f}  max|diff| {np.abs(g - r).max():.3e}")
    assert c >= 0.9999


@pytest.mark.parametrize("mode,name", [(1, "tanhf form"), (2, "ggml fp16 table")])
def test_so400m_vision_vs_reference_gelu_modes(orc, so400m_vision, mode, name):
    """The same embedding against the oracle with the reference CUDA
    epilogue's GELU formula (libm tanhf) and with ggml-cpu's fp16-table GELU
    (the reference's CPU path): the 0.9999 bar holds against both, the
    tower's differences from either being at the level of its own Q8_1
    rounding flips (measured 0.99995 for each)."""
    v, om = so400m_vision
    px = synth.pixels(1, 729, seed=1234)
    g = v.encode(px, 27, 27, s2x.POOL_PROBE)
    prev = orc.set_gelu_mode(mode)
    try:
        r = orc.vision_encode(om, px, 27, 27, pooling=1)
    finally:
        orc.set_gelu_mode(prev)
    c = cos(g, r)
    say(f"so400m vision 27x27 probe vs oracle GELU {name}: cosine {c:.7f}")
    assert c >= 0.9999


@pytest.mark.timeout(600)
def test_so400m_vision_batch_and_ragged_invariance(so400m_vision):
    v, _ = so400m_vision
    px = synth.pixels(4, 729, seed=77)
    b = v.batch(px, 4, 27, 27, s2x.POOL_PROBE)
    for i in (0, 3):
        one = v.batch(px[i * 729:(i + 1) * 729], 1, 27, 27, s2x.POOL_PROBE)
        assert np.array_equal(b[i], one[0])
    shapes = [(27, 27), (16, 16), (32, 32), (24, 24)]
    padded = np.zeros((4, 1024, 768), np.float32)
    singles = []
    for i, (h, w) in enumerate(shapes):
        p = synth.pixels(1, h * w, seed=300 + i)
        padded[i, :h * w] = p
        singles.append(v.batch(p, 1, h, w, s2x.POOL_PROBE)[0])
    out = v.ragged(padded.reshape(-1, 768), shapes, 1024, s2x.POOL_PROBE)
    for i in range(4):
        assert np.array_equal(out[i], singles[i])


@pytest.mark.timeout(600)
def test_so400m_vision_split_k(orc, so400m_vision):
    # the K-split GEMM option for batch-1 latency: an image's bits do not
    # depend on its batch with the option on, graph replays follow the
    # option as it is set, and the embedding stays within the tower's
    # sensitivity of the block-order oracle (each split GEMM is bit-exact
    # against its oracle restatement in test_gemm_split_k_bit_exact)
    v, om = so400m_vision
    px = synth.pixels(3, 729, seed=4321)
    plain = v.encode(px[:729], 27, 27, s2x.POOL_PROBE)
    s2x.call("s2x_vision_set_split_k", v.h, 1)
    try:
        # eager, captured, replayed
        split = [v.encode(px[:729], 27, 27, s2x.POOL_PROBE) for _ in range(3)]
        assert all(np.array_equal(split[0], g) for g in split[1:])
        assert not np.array_equal(split[0], plain)
        b = v.batch(px, 3, 27, 27, s2x.POOL_PROBE)
        assert np.array_equal(b[0], split[0])
        assert np.array_equal(b[2], v.batch(px[2 * 729:], 1, 27, 27, s2x.POOL_PROBE)[0])
        r = orc.vision_encode(om, px[:729], 27, 27, pooling=1)
        c = cos(split[0], r)
        say(f"so400m vision 27x27, K-split GEMMs: cosine {c:.7f} (block order: {cos(plain, r):.7f})")
        assert c >= 0.9998
    finally:
        s2x.call("s2x_vision_set_split_k", v.h, 0)
    for _ in range(2):
        assert np.array_equal(v.encode(px[:729], 27, 27, s2x.POOL_PROBE), plain)


@pytest.mark.timeout(600)
def test_so400m_vision_naflex_vs_oracle(orc, so400m_vision):
    v, om = so400m_vision
    h, w = 16, 64
    px = synth.pixels(1, h * w, seed=55)
    g = v.encode(px, h, w, s2x.POOL_MEAN)
    r = orc.vision_encode(om, px, h, w, pooling=0)
    c = cos(g, r)
    say(f"so400m vision 16x64 mean: cosine {c:.7f}")
    assert c >= 0.9999


@pytest.mark.timeout(600)
def test_so400m_vision_batch32_workload(orc, so400m_vision):
    """32 images x 729 patches (GEMM M = 23,328), the throughput workload:
    each image's embedding equals that image encoded alone, bit for bit, and
    the first and last match the oracle."""
    v, om = so400m_vision
    n = 32
    px = synth.pixels(n, 729, seed=4000)
    say("so400m vision 32 x 729")
    b = v.batch(px, n, 27, 27, s2x.POOL_PROBE)
    for i in (0, 13, 31):
        one = v.batch(px[i * 729:(i + 1) * 729], 1, 27, 27, s2x.POOL_PROBE)
        assert np.array_equal(b[i], one[0]), f"image {i}"
    for i in (0, 31):
        r = orc.vision_encode(om, px[i * 729:(i + 1) * 729], 27, 27, pooling=1)
        c = cos(b[i], r)
        say(f"  image {i}: cosine {c:.7f}")
        assert c >= 0.9999


NAFLEX_GRIDS = {256: [(16, 16), (8, 32), (32, 8)], 576: [(24, 24), (16, 36), (36, 16), (18, 32)],
                729: [(27, 27)], 1024: [(32, 32), (16, 64), (64, 16)]}


@pytest.mark.timeout(600)
def test_so400m_vision_naflex16_workload(orc, so400m_vision):
    """NaFlex ragged batch: 16 images, 4 each of 256, 576, 729 and 1024
    patches in seeded order, grids of several aspect ratios, padded to 1024
    patches.  Each embedding equals the image encoded alone, bit for bit;
    the widest and a 256-patch image match the oracle."""
    v, om = so400m_vision
    rng = np.random.default_rng(5000)
    counts = rng.permutation([256, 576, 729, 1024] * 4)
    shapes = [NAFLEX_GRIDS[c][rng.integers(len(NAFLEX_GRIDS[c]))] for c in counts]
    say(f"so400m vision NaFlex 16: {shapes}")
    padded = np.zeros((16, 1024, 768), np.float32)
    pix = []
    for i, (h, w) in enumerate(shapes):
        p = synth.pixels(1, h * w, seed=5100 + i)
        padded[i, :h * w] = p
        pix.append(p)
    out = v.ragged(padded.reshape(-1, 768), shapes, 1024, s2x.POOL_PROBE)
    for i, (h, w) in enumerate(shapes):
        one = v.batch(pix[i], 1, h, w, s2x.POOL_PROBE)[0]
        assert np.array_equal(out[i], one), f"image {i} ({h}x{w})"
    wide = [i for i, s in enumerate(shapes) if s[0] != s[1] and s[0] * s[1] == 1024]
    small = [i for i, s in enumerate(shapes) if s[0] * s[1] == 256]
    for i in (wide + [int(np.argmax(counts))])[:1] + small[:1]:
        h, w = shapes[i]
        r = orc.vision_encode(om, pix[i], h, w, pooling=1)
        c = cos(out[i], r)
        say(f"  image {i} ({h}x{w}): cosine {c:.7f}")
        assert c >= 0.9999


@pytest.mark.timeout(600)
def test_so400m_text_split_k(orc):
    # the K-split GEMM option: a prompt's bits do not depend on its batch;
    # against the block-order oracle the 27 random-weight layers amplify the
    # new summation order to cosine ~0.99988 (the tower's sensitivity, not an
    # error of the split: each split GEMM is bit-exact against its oracle
    # restatement in test_gemm_split_k_bit_exact)
    hm = synth.text_model(synth.SO400M_TEXT, seed=0)
    t = Text(hm)
    try:
        s2x.call("s2x_text_set_split_k", t.h, 1)
        om = orc.text_model(hm)
        ids, _ = synth.text_tokens(5, 64)
        b = t.batch(ids)
        assert np.array_equal(t.encode(ids[3]), b[3])
        c = cos(b[0], orc.text_encode(om, ids[0]))
        say(f"so400m text, K-split GEMMs: cosine {c:.7f}")
        assert c >= 0.9998
    finally:
        t.close()


@pytest.mark.timeout(600)
def test_so400m_text_5x64_vs_oracle(orc):
    say("generating so400m text weights")
    hm = synth.text_model(synth.SO400M_TEXT, seed=0)
    t = Text(hm)
    try:
        om = orc.text_model(hm)
        ids, _ = synth.text_tokens(5, 64)
        b = t.batch(ids)
        for i in (0, 4):
            r = orc.text_encode(om, ids[i])
            c = cos(b[i], r)
            say(f"so400m text prompt {i}: cosine {c:.7f}")
            assert c >= 0.9999
    finally:
        t.close()


def test_f16_ffn_down_forms_agree(orc):
    # fc2 of an F16 file with its bias and residual in the three tile forms of
    # the F16 GEMM (1, 4 and 32 images): the same bits, near the oracle
    cfg = synth.VisionConfig(n_layer=1)
    assert (cfg.hidden, cfg.inter) == (1152, 4304)
    hm = synth.vision_model(cfg, seed=27, down_f16=True)
    v = Vision(hm)
    try:
        px = synth.pixels(4, 729, seed=28)
        images = {f: rows // 729 for f, rows in F16_TOWER_ROWS.items()}
        say(f"F16 ffn_down forms: {images}")
        alone = np.concatenate([v.batch(px[i * 729:(i + 1) * 729], images["Small"], 27, 27, s2x.POOL_PROBE)
                                for i in range(4)])
        mid = v.batch(px, images["Mid"], 27, 27, s2x.POOL_PROBE)
        wide = v.batch(np.tile(px, (8, 1)), images["Wide"], 27, 27, s2x.POOL_PROBE)
    finally:
        v.close()
    assert np.array_equal(mid, alone)
    assert np.array_equal(wide, np.tile(alone, (8, 1)))
    ref = orc.vision_encode(orc.vision_model(hm), px[:729], 27, 27, pooling=s2x.POOL_PROBE)
    c = cos(alone[0], ref)
    say(f"  cosine vs oracle {c:.7f}")
    assert c >= 0.9999


def test_small_towers_f16_ffn_down(orc, tmp_path):
    """ffn_down as F16 (the converter's layout for K % 32 != 0): both towers
    against the oracle's F16 linear, batch / single invariance, and the
    towers created from a GGUF file of that layout give the same bits."""
    from gguf_util import text_tensors, vision_tensors, write_gguf
    hm = synth.vision_model(SMALL_V, seed=24, down_f16=True)
    v = Vision(hm)
    try:
        om = orc.vision_model(hm)
        px = synth.pixels(2, 729, seed=25)
        b = v.batch(px, 2, 27, 27, s2x.POOL_PROBE)
        for i in range(2):
            c = cos(b[i], orc.vision_encode(om, px[i * 729:(i + 1) * 729], 27, 27, pooling=1))
            say(f"small vision F16 ffn_down image {i}: cosine {c:.7f}")
            assert c >= 0.9999
        assert np.array_equal(v.batch(px[729:], 1, 27, 27, s2x.POOL_PROBE)[0], b[1])
        path = tmp_path / "v16.gguf"
        write_gguf(path, *vision_tensors(hm))
        g = ctypes.c_void_p()
        s2x.call("s2x_gguf_open", str(path).encode(), ctypes.byref(g))
        try:
            w = s2x.VisionWeights()
            s2x.call("s2x_gguf_vision_weights", g, ctypes.byref(w))
            assert w.down_f16 == 1
            h = ctypes.c_void_p()
            s2x.call("s2x_vision_create", ctypes.byref(w), ctypes.byref(h))
        finally:
            s2x.lib.s2x_gguf_close(g)
        try:
            pd = dev(px)
            out = empty((2, SMALL_V.hidden), torch.float32)
            s2x.call("s2x_vision_encode_batch_dev", h, ptr(pd), 2, 27, 27, s2x.POOL_PROBE, ptr(out))
            assert np.array_equal(host(out), b)
        finally:
            s2x.lib.s2x_vision_destroy(h)
    finally:
        v.close()

    hm = synth.text_model(SMALL_T, seed=26, down_f16=True)
    t = Text(hm)
    try:
        om = orc.text_model(hm)
        ids, _ = synth.text_tokens(3, 64, vocab=SMALL_T.vocab, seed=27)
        b = t.batch(ids)
        for i in range(3):
            c = cos(b[i], orc.text_encode(om, ids[i]))
            say(f"small text F16 ffn_down prompt {i}: cosine {c:.7f}")
            assert c >= 0.9999
            assert np.array_equal(t.encode(ids[i]), b[i])
        path = tmp_path / "t16.gguf"
        write_gguf(path, *text_tensors(hm))
        g = ctypes.c_void_p()
        s2x.call("s2x_gguf_open", str(path).encode(), ctypes.byref(g))
        try:
            w = s2x.TextWeights()
            s2x.call("s2x_gguf_text_weights", g, ctypes.byref(w))
            assert w.down_f16 == 1
            h = ctypes.c_void_p()
            s2x.call("s2x_text_create", ctypes.byref(w), ctypes.byref(h))
        finally:
            s2x.lib.s2x_gguf_close(g)
        try:
            out = np.empty((3, SMALL_T.proj), np.float32)
            s2x.call("s2x_text_encode_batch", h, ids.ctypes.data, 64, 3, out.ctypes.data)
            assert np.array_equal(out, b)
        finally:
            s2x.lib.s2x_text_destroy(h)
    finally:
        t.close()


def test_small_towers_from_gguf_same_bits(tmp_path, small_vision):
    """Encoders created from a GGUF file (s2x_gguf_*) equal the ones created
    from the host structs, bit for bit."""
    from gguf_util import text_tensors, vision_tensors, write_gguf
    v, _ = small_vision
    path = tmp_path / "v.gguf"
    write_gguf(path, *vision_tensors(v.host))
    g = ctypes.c_void_p()
    s2x.call("s2x_gguf_open", str(path).encode(), ctypes.byref(g))
    try:
        w = s2x.VisionWeights()
        s2x.call("s2x_gguf_vision_weights", g, ctypes.byref(w))
        h = ctypes.c_void_p()
        s2x.call("s2x_vision_create", ctypes.byref(w), ctypes.byref(h))
    finally:
        s2x.lib.s2x_gguf_close(g)  # the encoder holds device copies
    try:
        px = synth.pixels(2, 16 * 20, seed=91)
        pd = dev(px)
        out = empty((2, v.host.cfg.hidden), torch.float32)
        s2x.call("s2x_vision_encode_batch_dev", h, ptr(pd), 2, 16, 20, s2x.POOL_PROBE, ptr(out))
        assert np.array_equal(host(out), v.batch(px, 2, 16, 20, s2x.POOL_PROBE))
    finally:
        s2x.lib.s2x_vision_destroy(h)

    hm = synth.text_model(SMALL_T, seed=23)
    tpath = tmp_path / "t.gguf"
    write_gguf(tpath, *text_tensors(hm))
    ids, _ = synth.text_tokens(3, 64, vocab=SMALL_T.vocab, seed=9)
    outs = []
    for src in ("struct", "gguf"):
        h = ctypes.c_void_p()
        if src == "struct":
            s2x.call("s2x_text_create", ctypes.byref(hm.struct), ctypes.byref(h))
        else:
            s2x.call("s2x_gguf_open", str(tpath).encode(), ctypes.byref(g))
            try:
                w = s2x.TextWeights()
                s2x.call("s2x_gguf_text_weights", g, ctypes.byref(w))
                s2x.call("s2x_text_create", ctypes.byref(w), ctypes.byref(h))
            finally:
                s2x.lib.s2x_gguf_close(g)
        try:
            o = np.empty((3, SMALL_T.proj), np.float32)
            ids32 = np.ascontiguousarray(ids, np.int32)
            s2x.call("s2x_text_encode_batch", h, ids32.ctypes.data, 64, 3, o.ctypes.data)
            outs.append(o)
        finally:
            s2x.lib.s2x_text_destroy(h)
    assert np.array_equal(outs[0], outs[1])
