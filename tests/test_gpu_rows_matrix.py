"""The row-batched kernels that split a chain's products from its adds.

Few rows (k_chain_gemm): row counts around its 8-row tiles, outputs and K
that are no multiple of its tiles, with and without the fused norm and the
gate.  GEMMs on the matrix cores (k_mgemm): sizes that are no multiple of any
tile in rows, outputs or K, weights with signed zeros, sums that are flushed
to -0, subnormal weights, NaNs and infinities; against the vector-unit kernel
(CIS2_BGEMM16=0) and the oracle.  Prefill attention
(k_attention_tiles): every number of heads per item, runs that end inside a
tile, lengths around the 16-, 64- and 256-position steps, a cache end inside
a 16-position group, V rows with infinities and NaN past a row's own
position; against the per-row kernel (CIS2_ATT_TILES=0) and the oracle.
Attention of many decode rows (k_attention_wave).  The tree order of both:
reductions that end inside a block of 32 and inside a staged chunk, K long
enough that a partial block's zeros meet signed zeros.  The arithmetic is pinned,
so there is no tolerance."""
import os

import numpy as np
import pytest

import _oracle as O
from cis2amd import Cis2Model, artifacts

pytestmark = pytest.mark.gpu

ODD = artifacts.ModelSpec("odd", 132, 268, 1, 6, 2, 301, 1e-5, 10000.0, True, head_dim=22)
# K = 20 (one partial group of 16 and one of 4), a vocabulary of many tiles
WIDE = artifacts.ModelSpec("wide-vocab", 20, 28, 1, 2, 1, 40003, 1e-5, 10000.0, True)


# reductions of 260, 264 and 516: a partial 64-k slot; outputs that end inside
# an 8-row tile
FEW = artifacts.ModelSpec("few", 260, 516, 2, 4, 1, 301, 1e-5, 10000.0, True, head_dim=66)
# whole slots, q/k/v biases
FEW_QWEN2 = artifacts.ModelSpec("few-qwen2", 320, 256, 1, 5, 5, 97, 1e-6, 10000.0, True,
                                qkv_bias=True)


class EdgeWeights(artifacts.Weights):
    """The seeded weights with one entry in 16 replaced by +-0 and one in 16
    by +-2^-125 (in sums of ordinary size; Extremes has the sums that a
    product not flushed would change)."""

    def __init__(self, spec, seed):
        super().__init__(spec, seed)
        rng = np.random.default_rng(seed)
        for name, _, arr in self.tensors:
            if not name.endswith("norm.weight"):
                k = rng.integers(0, 16, arr.size)
                arr[k == 0] &= 0x8000
                arr[k == 1] = (arr[k == 1] & 0x8000) | 0x0100


def run(m, n, per_seq, tok, mode):
    os.environ["CIS2_BGEMM16"] = mode
    try:
        i = np.arange(n)
        lg, am = m.forward_rows(i // per_seq, i % per_seq, tok)
    finally:
        del os.environ["CIS2_BGEMM16"]
    return lg.view(np.uint32), am


@pytest.mark.parametrize("spec,n,per_seq", [
    (FEW, 1, 1),
    (FEW, 3, 1),         # one row per sequence (a decode step)
    (FEW, 8, 4),
    (FEW, 9, 9),
    (FEW, 31, 16),
    (FEW_QWEN2, 7, 7),
    (FEW_QWEN2, 17, 1),
    (WIDE, 5, 5),        # LM head: 64 x 16 tiles, one partial
    (WIDE, 16, 4),
    (WIDE, 17, 17),      # the first row count of the 32 x 32 tiles
    (ODD, 931, 19),      # 32 x 32 tiles, the last with 3 rows
    (ODD, 16001, 40),    # 64 x 64 tiles, the last with one row
], ids=lambda v: getattr(v, "name", str(v)))
def test_rows_matrix_core_gemm_bits(spec, n, per_seq):
    w = EdgeWeights(spec, 11)
    nseq = (n + per_seq - 1) // per_seq
    m = Cis2Model(spec, w, max_pos=per_seq, max_seqs=nseq)
    tok = np.random.default_rng(n).integers(0, spec.vocab, n).astype(np.uint32)
    lg, am = run(m, n, per_seq, tok, "1")
    lv, av = run(m, n, per_seq, tok, "0")
    assert np.array_equal(lg, lv)
    assert np.array_equal(am, av)
    for s in (0, nseq - 1):
        o = O.OracleModel(spec, w, max_pos=per_seq, reduction=0)
        for p in range(min(per_seq, n - s * per_seq)):
            want = o.forward(p, int(tok[s * per_seq + p])).view(np.uint32)
            assert np.array_equal(want, lg[s * per_seq + p]), (s, p)


def heads_spec(nh, nkv, hd):
    return artifacts.ModelSpec("h%d-%d-%d" % (nh, nkv, hd), 64, 64, 1, nh, nkv, 67, 1e-6, 10000.0,
                               True, head_dim=hd, qk_norm=hd == 128, sigma=0.3)


def tile_rows(lens):
    seq = np.repeat(np.arange(len(lens)), lens)
    return seq, np.concatenate([np.arange(n) for n in lens])


@pytest.mark.parametrize("nh,nkv,hd", [(1, 1, 64), (4, 2, 64), (3, 1, 64), (4, 1, 64), (5, 1, 64),
                                       (2, 2, 128), (2, 1, 128), (3, 1, 128), (4, 1, 128)])
@pytest.mark.parametrize("copies", [1, 300], ids=["one-head-items", "grouped-items"])
def test_attention_tiles_bits(nh, nkv, hd, copies):
    """copies = 300: enough tiles that an item takes the heads of a KV head
    together and a workgroup walks several items."""
    spec = heads_spec(nh, nkv, hd)
    w = artifacts.Weights(spec, 5)
    lens = [1, 17, 63, 66, 129, 259] if copies == 1 else [19, 34] * (copies // 2)
    m = Cis2Model(spec, w, max_pos=max(lens), max_seqs=len(lens))
    seq, pos = tile_rows(lens)
    tok = np.random.default_rng(3).integers(0, spec.vocab, seq.size).astype(np.uint32)
    out = {}
    for v in "01":
        os.environ["CIS2_ATT_TILES"] = v
        try:
            out[v], _ = m.forward_rows(seq, pos, tok)
        finally:
            del os.environ["CIS2_ATT_TILES"]
    assert np.array_equal(out["0"].view(np.uint32), out["1"].view(np.uint32))
    s = len(lens) - 1
    o = O.OracleModel(spec, w, max_pos=lens[s], reduction=0)
    rows = np.flatnonzero(seq == s)
    for p, r in enumerate(rows):
        assert np.array_equal(o.forward(p, int(tok[r])).view(np.uint32),
                              out["1"][r].view(np.uint32)), p


@pytest.mark.parametrize("nh,nkv,hd", [(3, 1, 64), (2, 2, 64), (2, 1, 128), (5, 5, 128)])
@pytest.mark.parametrize("pos", [0, 2, 63, 64, 130])
def test_attention_wave_bits(nh, nkv, hd, pos):
    """Decode rows of so many sequences that a wave takes each (row, head),
    RoPE and cache stores in the same launch: logits equal to the
    one-workgroup kernel's (CIS2_ATT_KV=0) for this step and the next, which
    reads what the first one stored, and to the oracle's."""
    spec = heads_spec(nh, nkv, hd)
    n = 2100 // nh
    w = artifacts.Weights(spec, 8)
    m = Cis2Model(spec, w, max_pos=pos + 2, max_seqs=n)
    tok = np.random.default_rng(4).integers(0, spec.vocab, (n, pos + 2)).astype(np.uint32)
    out = {}
    for v in ("0", "256"):
        os.environ["CIS2_ATT_KV"] = v
        try:
            if pos:
                m.forward_rows(np.repeat(np.arange(n), pos), np.tile(np.arange(pos), n),
                               tok[:, :pos].reshape(-1), want_logits=False)
            out[v] = [m.forward_rows(np.arange(n), np.full(n, p), tok[:, p])[0]
                      for p in (pos, pos + 1)]
        finally:
            del os.environ["CIS2_ATT_KV"]
    for a, b in zip(out["0"], out["256"]):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    o = O.OracleModel(spec, w, max_pos=pos + 2, reduction=0)
    for p in range(pos + 2):
        want = o.forward(p, int(tok[n - 1, p]))
    assert np.array_equal(want.view(np.uint32), out["256"][1][n - 1].view(np.uint32))


def test_attention_tiles_later_rows_do_not_leak():
    """A row whose V (and K) hold NaN or infinities changes no row before it,
    also inside one tile; it and the rows after it get the per-row kernel's
    bits, those of the NaNs among them."""
    spec = heads_spec(2, 1, 64)
    w = artifacts.Weights(spec, 6)
    emb = next(a for name, _, a in w.tensors if "embed" in name)
    emb[7 * spec.hidden] = 0x7F80       # token 7: +inf in one dimension
    emb[8 * spec.hidden + 1] = 0xFFC1   # token 8: a NaN
    n = 41
    tok = np.arange(20, 20 + n).astype(np.uint32)
    clean = Cis2Model(spec, w, max_pos=n)
    base, _ = clean.forward_rows(np.zeros(n), np.arange(n), tok)
    for at, bad in ((5, 7), (18, 8), (40, 7)):
        t2 = tok.copy()
        t2[at:at + 1] = bad
        os.environ["CIS2_ATT_TILES"] = "1"
        try:
            got, _ = clean.forward_rows(np.zeros(n), np.arange(n), t2)
        finally:
            del os.environ["CIS2_ATT_TILES"]
        assert np.array_equal(got[:at].view(np.uint32), base[:at].view(np.uint32)), at
        assert not np.isfinite(got[at]).all()
        os.environ["CIS2_ATT_TILES"] = "0"
        try:
            rows, _ = clean.forward_rows(np.zeros(n), np.arange(n), t2)
        finally:
            del os.environ["CIS2_ATT_TILES"]
        assert np.isnan(rows[at:]).any()
        assert np.array_equal(got.view(np.uint32), rows.view(np.uint32)), at  # NaNs' bits too


def tree_model(spec, w, per_seq, nseq):
    return Cis2Model(spec, w, max_pos=per_seq, max_seqs=nseq, reduction_mode=1)


@pytest.mark.parametrize("spec,n,per_seq", [
    (WIDE, 5, 5),        # LM head: 64 x 16 tiles, one partial, K = 20 of 32
    (WIDE, 17, 17),      # 32 x 32 tiles
    (ODD, 931, 19),      # K = 132 and 268: a block of 4 and one of 12
    (FEW, 300, 30),      # 260 and 516
    (FEW_QWEN2, 700, 50),
    (ODD, 16001, 40),    # 64 x 64 tiles, the last with one row
], ids=lambda v: getattr(v, "name", str(v)))
def test_tree_rows_matrix_core_gemm_bits(spec, n, per_seq):
    w = EdgeWeights(spec, 12)
    nseq = (n + per_seq - 1) // per_seq
    m = tree_model(spec, w, per_seq, nseq)
    tok = np.random.default_rng(n).integers(0, spec.vocab, n).astype(np.uint32)
    lg, am = run(m, n, per_seq, tok, "1")
    lv, av = run(m, n, per_seq, tok, "0")
    assert np.array_equal(lg, lv)
    assert np.array_equal(am, av)
    o = O.OracleModel(spec, w, max_pos=per_seq, reduction=1)
    first = (nseq - 1) * per_seq
    for p in range(n - first):
        want = o.forward(p, int(tok[first + p])).view(np.uint32)
        assert np.array_equal(want, lg[first + p]), p


@pytest.mark.parametrize("nh,nkv,hd", [(1, 1, 64), (4, 2, 64), (3, 1, 64), (2, 1, 128),
                                       (3, 1, 128)])
@pytest.mark.parametrize("copies", [1, 300], ids=["one-head-items", "grouped-items"])
def test_tree_attention_tiles_bits(nh, nkv, hd, copies):
    spec = heads_spec(nh, nkv, hd)
    w = artifacts.Weights(spec, 5)
    lens = [1, 17, 31, 33, 66, 129, 259] if copies == 1 else [19, 34] * (copies // 2)
    m = tree_model(spec, w, max(lens), len(lens))
    seq, pos = tile_rows(lens)
    tok = np.random.default_rng(3).integers(0, spec.vocab, seq.size).astype(np.uint32)
    out = {}
    for v in "01":
        os.environ["CIS2_ATT_TILES"] = v
        try:
            out[v], _ = m.forward_rows(seq, pos, tok)
        finally:
            del os.environ["CIS2_ATT_TILES"]
    assert np.array_equal(out["0"].view(np.uint32), out["1"].view(np.uint32))
    s = len(lens) - 1
    o = O.OracleModel(spec, w, max_pos=lens[s], reduction=1)
    for p, r in enumerate(np.flatnonzero(seq == s)):
        assert np.array_equal(o.forward(p, int(tok[r])).view(np.uint32),
                              out["1"][r].view(np.uint32)), p


def logits_spec(k, vocab=40003):
    return artifacts.ModelSpec("lm%d" % k, k, 72, 1, 2, 1, vocab, 1e-5, 10000.0, False)


class TinySums(artifacts.Weights):
    """The seeded weights, final norm weights of 2; an LM head row is +-0 but
    for one entry of 2^-126 .. 2^-122 in its first block of 32 and one at its
    end, so that among many rows some sums cancel to a negative value that is
    flushed, to -0."""

    def __init__(self, spec, seed):
        super().__init__(spec, seed)
        rng = np.random.default_rng(seed)
        h, v = spec.hidden, spec.vocab
        w = (rng.integers(0, 2, (v, h)) << 15).astype(np.uint16)
        for lo, hi in ((0, 32), (h - 1, h)):
            at = (np.arange(v), rng.integers(lo, hi, v))
            w[at] |= rng.integers(1 << 7, 5 << 7, v).astype(np.uint16)
        for name, _, arr in self.tensors:
            if name == "lm_head.weight":
                arr[:] = w.reshape(-1)
            elif name == "model.norm.weight":
                arr[:] = 0x4000


@pytest.mark.parametrize("tree", [True, False], ids=["tree", "seq"])
@pytest.mark.parametrize("k", [68, 96, 100, 132, 160])
@pytest.mark.parametrize("n", [5, 17])  # 64 x 16 and 32 x 32 tiles
def test_rows_matrix_core_gemm_negative_zero_sums(k, n, tree):
    """A sum of -0 stays -0 whatever lies between K and the end of the staged
    chunk (64 k: at K = 68, 96, 132 and 160 a whole block of 32 lies past K)."""
    spec = logits_spec(k)
    w = TinySums(spec, 13)
    m = Cis2Model(spec, w, max_pos=n, max_seqs=1, reduction_mode=1 if tree else 0)
    tok = np.random.default_rng(n).integers(0, spec.vocab, n).astype(np.uint32)
    lg, am = run(m, n, n, tok, "1")
    o = O.OracleModel(spec, w, max_pos=n, reduction=1 if tree else 0)
    want = np.stack([o.forward(p, int(tok[p])) for p in range(n)]).view(np.uint32)
    assert (want == 0x80000000).sum() > 1000
    assert np.array_equal(want, lg)
    lv, av = run(m, n, n, tok, "0")
    assert np.array_equal(want, lv)
    assert np.array_equal(am, av)


class Extremes(artifacts.Weights):
    """The seeded weights, final norm weights of 2^8; of every four LM head
    rows one holds subnormals only (times activations that would lift them
    far above 2^-126 if they were not flushed), one a NaN of any
    sign and payload among its values, one two infinities, one +-0 and entries
    whose products lie around 2^-126."""

    def __init__(self, spec, seed):
        super().__init__(spec, seed)
        rng = np.random.default_rng(seed)
        h, v = spec.hidden, spec.vocab
        for name, _, arr in self.tensors:
            if name == "model.norm.weight":
                arr[:] = 0x4380
            elif name == "lm_head.weight":
                w = arr.reshape(v, h)
                sign = (rng.integers(0, 2, (v, h)) << 15).astype(np.uint16)
                w[0::4] = (sign | rng.integers(1, 0x80, (v, h)).astype(np.uint16))[0::4]
                r = np.arange(1, v, 4)
                w[r, rng.integers(0, h, r.size)] = (0x7F81 + rng.integers(0, 0x7F, r.size) |
                                                   rng.integers(0, 2, r.size) << 15)
                r = np.arange(2, v, 4)
                for _ in range(2):
                    w[r, rng.integers(0, h, r.size)] = 0x7F80 | rng.integers(0, 2, r.size) << 15
                k = rng.integers(0, 5 << 7, (v, h)).astype(np.uint16)
                w[3::4] = (sign | np.where(rng.random((v, h)) < 0.5, k, 0).astype(np.uint16))[3::4]


@pytest.mark.parametrize("tree", [True, False], ids=["tree", "seq"])
@pytest.mark.parametrize("k", [20, 68])
@pytest.mark.parametrize("n", [5, 17])
def test_rows_matrix_core_gemm_subnormals_and_nans(k, n, tree):
    """The matrix cores' products flush subnormal operands and results and
    carry NaNs as the vector unit's multiply does: the bits of every logit,
    NaNs' sign and payload too, are the vector-unit kernel's, and those of
    every other logit the oracle's (NaNs made by x86 have another sign)."""
    spec = logits_spec(k)
    w = Extremes(spec, 14)
    m = Cis2Model(spec, w, max_pos=n, max_seqs=1, reduction_mode=1 if tree else 0)
    tok = np.random.default_rng(n).integers(0, spec.vocab, n).astype(np.uint32)
    lg, am = run(m, n, n, tok, "1")
    lv, av = run(m, n, n, tok, "0")
    assert np.array_equal(lg, lv)
    assert np.array_equal(am, av)
    o = O.OracleModel(spec, w, max_pos=n, reduction=1 if tree else 0)
    want = np.stack([o.forward(p, int(tok[p])) for p in range(n)])
    got = lg.view(np.float32)
    assert not want[:, 0::4].any()  # subnormal weights are zeros
    nan = np.isnan(want)
    assert nan[:, 1::4].all() and np.array_equal(nan, np.isnan(got))
    assert np.array_equal(want.view(np.uint32)[~nan], lg[~nan])


@pytest.mark.parametrize("tree", [True, False], ids=["tree", "seq"])
@pytest.mark.parametrize("hd", [6, 22, 34])
def test_qk_norm_of_head_dims_that_are_no_multiple_of_four(hd, tree):
    """The vectors of such a QK-norm take the norm kernel that has a workgroup
    per vector; many and few rows, and one position at a time."""
    spec = artifacts.ModelSpec("qk%d" % hd, 64, 96, 2, 4, 2, 131, 1e-6, 10000.0, True,
                               head_dim=hd, qk_norm=True, sigma=0.3)
    w = artifacts.Weights(spec, 15)
    n = 70
    tok = np.random.default_rng(hd).integers(0, spec.vocab, n).astype(np.uint32)
    o = O.OracleModel(spec, w, max_pos=n, reduction=1 if tree else 0)
    want = np.stack([o.forward(p, int(tok[p])) for p in range(n)]).view(np.uint32)
    m = Cis2Model(spec, w, max_pos=n, max_seqs=1, reduction_mode=1 if tree else 0)
    lg, _ = m.forward_rows(np.zeros(n), np.arange(n), tok)
    assert np.array_equal(want, lg.view(np.uint32))
    m.reset(0)
    for at, k in ((0, 1), (1, 3), (4, 1)):
        lg, _ = m.forward_rows(np.zeros(k), np.arange(at, at + k), tok[at:at + k])
        assert np.array_equal(want[at:at + k], lg.view(np.uint32)), at


@pytest.mark.parametrize("tree", [True, False], ids=["tree", "seq"])
@pytest.mark.parametrize("k,n", [(68, 40), (300, 17)])
def test_several_nans_keep_their_places(k, n, tree):
    """Where different NaNs and infinities meet in the sums, every path has
    the same NaN logits and the same bits in all others; in tree order the row
    GEMMs have the bits of the persistent kernel in the NaNs too (the left
    operand's)."""
    spec = artifacts.ModelSpec("nans%d" % k, k, 188, 2, 4, 2, 5003, 1e-5, 10000.0, False,
                               head_dim=64)
    w = artifacts.Weights(spec, 16)
    rng = np.random.default_rng(16)
    for name, _, arr in w.tensors:
        a, some = arr.reshape(-1), arr.size // 5000
        if "lm_head" in name:
            sign = rng.integers(0, 2, 2 * some) << 15
            a[rng.integers(0, a.size, some)] = 0x7F80 | sign[:some]
            a[rng.integers(0, a.size, some)] = 0x7FA1 + rng.integers(0, 30, some) | sign[some:]
            a[::7 * k] = 0xFFB1  # against the NaN activations of the first block
        elif "embed" in name:
            a[-k:][[0, 7, 8]] = [0x7FA1, 0xFFC2, 0xFF80]  # the last token's
    tok = rng.integers(0, spec.vocab - 1, n).astype(np.uint32)
    tok[n // 2] = spec.vocab - 1
    m = Cis2Model(spec, w, max_pos=n, max_seqs=1, reduction_mode=1 if tree else 0)
    rows, _ = run(m, n, n, tok, "1")
    vec, _ = run(m, n, n, tok, "0")
    m.reset(0)
    one = np.stack([m.forward_token(p, int(tok[p]))[0] for p in range(n)])
    nan = np.isnan(one)
    assert nan[n // 2].all() and nan[0].any() and not nan[:n // 2].all(axis=1).any()
    for got in (rows, vec):
        assert np.array_equal(np.isnan(got.view(np.float32)), nan)
        assert np.array_equal(got[~nan], one.view(np.uint32)[~nan])
        if tree:
            assert np.array_equal(got, one.view(np.uint32))
