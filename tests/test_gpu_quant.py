"""GPU producer parity: the synthetic generator and the codebook quantiser, bit-exact against the
reference's own outputs (golden fixtures written by the compiled reference) and the oracle."""
import hashlib
import json
import os

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")


def sha(a) -> str:
    return hashlib.sha256(np.ascontiguousarray(a).tobytes()).hexdigest()


@pytest.fixture(scope="module")
def ax():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import affinity_amd.experts as ax
    ax.init()
    return ax


def test_generator_matches_oracle(ax, orc):
    n = 1 << 22
    for seed, scale in ((1000, 0.02), (7, 1.0)):
        got = ax.gen_normal(seed, n, scale).cpu().numpy()
        ref = orc.normal_bf16(seed, n, scale)
        np.testing.assert_array_equal(got.view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("case", ["a", "b", "c", "d"])
def test_quantizer_matches_reference_small(ax, small, c1_codebook, case):
    cbf = torch.from_numpy(ax.codebook_floats(c1_codebook)).cuda()
    w = small[f"{case}_w"]
    gw = torch.from_numpy(w).cuda()
    codes, fields, rs = ax.quantize_matrix(gw, cbf)
    np.testing.assert_array_equal(codes.cpu().numpy(), small[f"{case}_codes"])
    np.testing.assert_array_equal(fields.cpu().numpy(), small[f"{case}_fields"])
    np.testing.assert_array_equal(rs.cpu().numpy().view(np.uint16), small[f"{case}_rs"])
    imp = torch.from_numpy(small[f"{case}_imp"]).cuda()
    codes, fields, _ = ax.quantize_matrix(gw, cbf, imp)
    np.testing.assert_array_equal(codes.cpu().numpy(), small[f"{case}_codes_imp"])
    np.testing.assert_array_equal(fields.cpu().numpy(), small[f"{case}_fields_imp"])


def test_quantizer_matches_reference_config1(ax, c1_codebook):
    """The config-1 expert quantised on the GPU has the reference's exact plane hashes."""
    man = json.load(open(os.path.join(GOLDEN, "c1_manifest.json")))
    cbf = torch.from_numpy(ax.codebook_floats(c1_codebook)).cuda()
    H, I = 4096, 2048
    for m, (name, rows, cols) in enumerate((("gate", I, H), ("up", I, H), ("down", H, I))):
        w = ax.gen_normal(1000 + m, rows * cols, 0.02).view(rows, cols)
        assert sha(w.cpu().numpy()) == man["inputs"][name]
        codes, fields, rs = ax.quantize_matrix(w, cbf)
        torch.cuda.synchronize()
        assert sha(codes.cpu().numpy()) == man["planes"][name]["codes"], name
        assert sha(fields.cpu().numpy()) == man["planes"][name]["fields"], name
        assert sha(rs.cpu().numpy().view(np.uint16)) == man["planes"][name]["rscales"], name


@pytest.mark.parametrize("rows,cols", [(3, 64), (2, 448), (5, 1088), (2, 8192)])
@pytest.mark.parametrize("kind", ["normal", "ties", "scales", "importance", "nonfinite", "codebook"])
def test_quantizer_edges_match_oracle(ax, orc, c1_codebook, rows, cols, kind):
    """Bit for bit against the oracle where the setting's choice is hard: a codebook whose settings tie
    (its second variant the first one negated, entries repeated), rows from 1e-42 to 1e38 with zero
    blocks, importances that are zero or negative, infinities and NaN in the rows or the codebook; partial chunks and a whole row of
    8192."""
    rng = np.random.default_rng(rows * cols + len(kind))
    w = (0.02 * rng.standard_normal((rows, cols))).astype(np.float32)
    cb = ax.codebook_floats(c1_codebook).copy()
    imp = None
    if kind == "ties":
        cb[1] = -cb[0]
        cb[:, 512:] = cb[:, :512]
        w[:, ::2] = np.sign(w[:, ::2]) * np.float32(0.0078125)
    elif kind == "scales":
        w[0] *= np.float32(1e-40)
        w[-1] *= np.float32(4e38 / 100)
        w[0, 16:32] = 0
        w[rows // 2, :64] = 0
        w[rows // 2, 5] = np.float32(3e3)
    elif kind == "importance":
        imp = rng.uniform(-0.2, 1.0, cols).astype(np.float32)
        imp[:32] = 0
        imp[32:64] = np.abs(imp[32:64])
    elif kind == "nonfinite":
        w[0, 7] = np.inf
        w[1, 20] = np.nan
        w[-1, 33] = -np.inf
    elif kind == "codebook":
        cb[0, 5], cb[0, 261, 2], cb[1, 900, 0] = 1e10, np.nan, -np.inf
    want = orc.quantize(w, cb.reshape(-1), imp)
    codes, fields, rs = ax.quantize_matrix(torch.from_numpy(w).cuda(), torch.from_numpy(cb).cuda(),
                                           None if imp is None else torch.from_numpy(imp).cuda())
    np.testing.assert_array_equal(rs.cpu().numpy().view(np.uint16), np.asarray(want[2]).view(np.uint16))
    np.testing.assert_array_equal(fields.cpu().numpy(), np.asarray(want[1]).view(np.uint8))
    np.testing.assert_array_equal(codes.cpu().numpy(), np.asarray(want[0]).view(np.uint8))


@pytest.mark.parametrize("tied", [False, True])
@pytest.mark.parametrize("wscale,cscale,iscale,spike", [
    (1e-20, 1e-5, 0, 0), (1e-22, 1e-3, 0, 0), (1e-24, 1e-5, 0, 0), (1e-26, 1e-5, 0, 0), (1e-28, 1.0, 0, 0),
    (1.0, 0.0039, 0, 0), (1e-21, 1e-21, 0, 1), (1e-19, 1e-19, 0, 1), (1.0, 1e-12, 0, 0), (1.0, 1.0, 1e-40, 0),
    (1.0, 1.0, 1e-28, 0), (1.0, 1.0, 1e12, 0)])
def test_quantizer_underflow_matches_oracle(ax, orc, c1_codebook, wscale, cscale, iscale, spike, tied):
    """Bit for bit against the oracle where squares, distances or weighted sums underflow: rows and
    codebooks scaled down together and apart (tied: the second variant the first one negated),
    blocks far below the row's scale (spike: its last weight), importances near zero."""
    rng = np.random.default_rng(77)
    rows, cols = 24, 1024
    w = (np.float32(wscale) * (0.02 * rng.standard_normal((rows, cols)))).astype(np.float32)
    if spike:
        w[:, -1] = spike
    cb = (ax.codebook_floats(c1_codebook) * np.float32(cscale)).astype(np.float32)
    if tied:
        cb[1] = -cb[0]
    imp = (np.float32(iscale) * rng.uniform(0.1, 1.1, cols)).astype(np.float32) if iscale else None
    want = orc.quantize(w, cb.reshape(-1), imp)
    codes, fields, rs = ax.quantize_matrix(torch.from_numpy(w).cuda(), torch.from_numpy(cb).cuda(),
                                           None if imp is None else torch.from_numpy(imp).cuda())
    np.testing.assert_array_equal(rs.cpu().numpy().view(np.uint16), np.asarray(want[2]).view(np.uint16))
    np.testing.assert_array_equal(fields.cpu().numpy(), np.asarray(want[1]).view(np.uint8))
    np.testing.assert_array_equal(codes.cpu().numpy(), np.asarray(want[0]).view(np.uint8))


@pytest.mark.parametrize("cols", [64, 128, 512, 1088])
def test_quantizer_open_blocks_match_oracle(ax, orc, c1_codebook, cols):
    """Every block left to the full search, shared among a workgroup's waves: importances below zero,
    all zero, and (with importances) blocks of zeros between; rows of one short chunk."""
    rng = np.random.default_rng(cols)
    rows = 12
    w = (0.02 * rng.standard_normal((rows, cols))).astype(np.float32)
    w[1, 16:32] = 0
    w[2] = 0
    cb = ax.codebook_floats(c1_codebook)
    gw, gc = torch.from_numpy(w).cuda(), torch.from_numpy(cb).cuda()
    for imp in (rng.uniform(-1.0, 0.2, cols).astype(np.float32), np.zeros(cols, np.float32)):
        want = orc.quantize(w, cb.reshape(-1), imp)
        codes, fields, rs = ax.quantize_matrix(gw, gc, torch.from_numpy(imp).cuda())
        np.testing.assert_array_equal(fields.cpu().numpy(), np.asarray(want[1]).view(np.uint8))
        np.testing.assert_array_equal(codes.cpu().numpy(), np.asarray(want[0]).view(np.uint8))
        np.testing.assert_array_equal(rs.cpu().numpy().view(np.uint16), np.asarray(want[2]).view(np.uint16))


@pytest.mark.parametrize("rows,cols", [(5, 64), (768, 128), (769, 128)])
def test_quantizer_short_rows_match_oracle(ax, orc, c1_codebook, rows, cols):
    """Rows of 64 and 128 columns, bit for bit, on both sides of the row count from which those of 128 are
    searched in full; with and without importances, with rows and blocks of zeros."""
    rng = np.random.default_rng(rows)
    w = (0.02 * rng.standard_normal((rows, cols))).astype(np.float32)
    w[1, 16:32] = 0
    w[2] = 0
    cb = ax.codebook_floats(c1_codebook)
    for imp in (None, rng.uniform(0.1, 1.1, cols).astype(np.float32)):
        want = orc.quantize(w, cb.reshape(-1), imp)
        codes, fields, rs = ax.quantize_matrix(torch.from_numpy(w).cuda(), torch.from_numpy(cb).cuda(),
                                               None if imp is None else torch.from_numpy(imp).cuda())
        np.testing.assert_array_equal(rs.cpu().numpy().view(np.uint16), np.asarray(want[2]).view(np.uint16))
        np.testing.assert_array_equal(fields.cpu().numpy(), np.asarray(want[1]).view(np.uint8))
        np.testing.assert_array_equal(codes.cpu().numpy(), np.asarray(want[0]).view(np.uint8))
