"""The down projection: sizes at the edges of its row blocks, stages and column shares; z with single large values, and with values
that are not finite."""
import numpy as np
import pytest

import helpers
from oracle import ref_oracle as o

pytestmark = pytest.mark.gpu

# one expert per count: edges of the 16-row blocks, of the 16-assignment chunks, of the 64- and 128-row tiles
COUNTS = (1, 15, 16, 17, 32, 33, 64, 65, 129)


def _run(cuda_device, gate, up, down, h_gate, h_up, tok, off, rw, rank_out, dim, path):
    import torch
    from bitsmoe_amd.algorithms import mlp_forward_cuda as hip

    sets = [hip.MatrixSet(*helpers.to_device_lists(m, cuda_device), intermediate_size=dim) for m in (gate, up, down)]
    dev = [torch.from_numpy(x).to(cuda_device) for x in (tok, off, rw)]
    return hip.moe_forward_sets(h_gate.to(cuda_device), h_up.to(cuda_device), *dev, *sets, rank_out, dim, 0, path=path).cpu().numpy()


def _inputs(seed, dim, choices, counts=COUNTS, rank=192):
    import torch

    rng = np.random.default_rng(seed)
    n = len(counts)
    gate, up, down = helpers.make_experts(seed, n, rank, rank, dim, choices=choices, uniform_bits=len(choices) == 1)
    tokens = max(counts)
    tok = np.concatenate([rng.permutation(tokens)[:c] for c in counts]).astype(np.int32)
    off = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    rw = rng.uniform(0.1, 1.0, size=tok.size).astype(np.float32)
    h = [torch.from_numpy(rng.normal(size=(tokens, rank)).astype(np.float32)).to(torch.bfloat16) for _ in range(2)]
    return gate, up, down, *h, tok, off, rw, rank


@pytest.mark.parametrize("dim", [128, 896, 1920])      # one tile; shares of four and three tiles at decode; fifteen tiles
@pytest.mark.parametrize("choices", [(2,), (3,), (4,), (2, 3, 4)])
@pytest.mark.parametrize("path_name", ["decode", "mfma"])
def test_rows_at_the_edges_of_blocks_and_tiles(cuda_device, path_name, choices, dim):
    from bitsmoe_amd.algorithms import _capi

    gate, up, down, h_gate, h_up, tok, off, rw, rank = _inputs(dim + len(choices), dim, choices)
    got = _run(cuda_device, gate, up, down, h_gate, h_up, tok, off, rw, rank, dim,
               _capi.PATH_MFMA if path_name == "mfma" else _capi.PATH_DECODE)
    ref = o.moe_forward(h_gate.float().numpy(), h_up.float().numpy(), tok, off, rw, gate, up, down, rank, dim)
    # an operand of gate, of up, their sums (grouped GEMM) and z are each rounded once to f16: at most 2^-11 of a value each
    assert helpers.norm_err(got, ref) <= 5 * 2.0 ** -11


@pytest.mark.parametrize("path_name", ["decode", "mfma"])
def test_a_token_that_is_not_finite_stays_by_itself(cuda_device, path_name):
    """A token whose z is not finite has outputs that are not finite.  The tokens that share its row blocks, tiles and experts are what
    they are without it."""
    from bitsmoe_amd.algorithms import _capi

    path = _capi.PATH_MFMA if path_name == "mfma" else _capi.PATH_DECODE
    gate, up, down, h_gate, h_up, tok, off, rw, rank = _inputs(7, 256, (2, 3, 4), counts=(20, 20, 20))
    clean = _run(cuda_device, gate, up, down, h_gate, h_up, tok, off, rw, rank, 256, path)
    assert np.isfinite(clean).all()
    for bad in (np.inf, np.nan):
        h_bad = h_up.clone()
        h_bad[5] = bad
        got = _run(cuda_device, gate, up, down, h_gate, h_bad, tok, off, rw, rank, 256, path)
        assert not np.isfinite(got[5]).any()
        others = np.arange(20) != 5
        assert np.allclose(got[others], clean[others], rtol=0, atol=1e-5 * np.abs(clean).max())      # (order of the atomics)


def _z_with_large_columns(seed, counts, large_up, large_gate, down_choices, dim=256, rank=192):
    """Experts with one column of z = silu(G) * U in 32 larger than the others: activations of one sign, and there a weight of one
    sign and size (0: as everywhere) in all rows of up and gate.  The first half of the down rows has level zero in these columns."""
    import torch

    rng = np.random.default_rng(seed)
    large = np.arange(dim) % 32 == 5
    gate, up, down = [], [], []
    for _ in counts:
        for lst, size in ((gate, large_gate), (up, large_up)):
            w = rng.normal(0.0, 0.02, size=(rank, dim)).astype(np.float32)
            if size:
                w[:, large] = size
            lst.append(o.pack_matrix(w, np.ones(rank, np.float32), [(4, (0, rank))]))
        w = rng.normal(0.0, 0.02, size=(rank, dim)).astype(np.float32)
        w[: rank // 2, large] = 0.0
        cuts = [0, 40, 130, rank]
        segments = [(b, (r0, r1)) for b, r0, r1 in zip(down_choices, cuts[:-1], cuts[1:])]
        down.append(o.pack_matrix(w, np.ones(rank, np.float32), segments))
    tokens = max(counts)
    tok = np.concatenate([rng.permutation(tokens)[:c] for c in counts]).astype(np.int32)
    off = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    rw = rng.uniform(0.1, 1.0, size=tok.size).astype(np.float32)
    h = [torch.from_numpy(0.3 + np.abs(rng.normal(size=(tokens, rank))).astype(np.float32)).to(torch.bfloat16) for _ in range(2)]
    return gate, up, down, *h, tok, off, rw, rank


# rms of rounding to eleven bits, over a binade
ROUNDING = 2.0 ** -11 / (3.0 * 2.0) ** 0.5


@pytest.mark.parametrize("large", [(0.0, 0.0), (0.1, 0.0), (0.1, 0.02)])      # 1, about 60 and about 1000 times the others
@pytest.mark.parametrize("down_choices", [(2, 2, 2), (3, 3, 3), (2, 4, 3), (2, 8, 16)])
@pytest.mark.parametrize("path_name,counts", [("mfma", (20, 33, 64)), ("decode", (20, 17, 16)), ("decode", (2, 1, 3)),
                                              ("decode", (0, 0, 2, 0, 0, 0, 1, 0))])      # chunks, experts, active experts
def test_small_columns_of_z_beside_large_ones(cuda_device, path_name, counts, down_choices, large):
    """Outputs whose weights at the large columns are zero see the small ones alone: every element of z has an f16 number's bits,
    however large its neighbours are."""
    from bitsmoe_amd.algorithms import _capi

    gate, up, down, h_gate, h_up, tok, off, rw, rank = _z_with_large_columns(sum(counts), counts, *large, down_choices)
    got = _run(cuda_device, gate, up, down, h_gate, h_up, tok, off, rw, rank, 256,
               _capi.PATH_MFMA if path_name == "mfma" else _capi.PATH_DECODE)
    ref = o.moe_forward(h_gate.float().numpy(), h_up.float().numpy(), tok, off, rw, gate, up, down, rank, 256)
    small = slice(0, rank // 2)
    err = np.linalg.norm(got[:, small] - ref[:, small]) / np.linalg.norm(ref[:, small])
    # at most six independent roundings of that size: the operands of gate, up and down, both sums and z; twice that for the
    # sums' own spread over a few tokens
    assert err <= 2 * 6 ** 0.5 * ROUNDING, f"{err:.3e}"
