"""The down projection's z as three fp6 planes against the packed codes (csrc/z_planes.h): sizes at the edges of its row blocks,
stages and column shares, and values that a plane cannot hold."""
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
    """z without a finite value has no planes: its block's scale is the format's NaN, and the token's outputs are not finite.  The
    tokens that share its row blocks, tiles and experts are what they are without it."""
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
