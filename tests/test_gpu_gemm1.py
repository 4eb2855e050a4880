"""SwiGLU rows of GEMM1 where an expert's row count picks the tile (up to 128
rows, 256 rows, remainders of both), against the CPU oracle, on either side of
the token count where the wide tiles start."""
import numpy as np
import pytest
import torch

from test_gpu_gemm2 import tokens_with_rows
from test_gpu_layer import run_layer
from util import bf16_close, gpu_weights, oracle_inputs

pytestmark = pytest.mark.gpu

# one token's picks stay within 8: the counts sum to at most 8 T
COUNTS = (1, 63, 64, 65, 127, 128, 129, 192, 193, 255, 256, 257, 384, 385, 513, 16)


def check_rows(pkg, orc, cuda_device, T, counts):
    """Experts 0 .. len(counts) - 1 with counts[e] rows each: act rows at the
    edges of every 64 rows against the oracle."""
    cfg = pkg.synth.CONFIGS["prefill_t1024"]
    w, w_host = gpu_weights(pkg, cfg.seed, cuda_device)
    tok, host = tokens_with_rows(pkg, cfg, cuda_device, T, counts)
    print(f"GEMM1 row counts T={T}", flush=True)
    run_layer(pkg, tok, w, 0, cfg.routed_scaling_factor)
    r = pkg.intermediates(pkg.workspace(cuda_device, T), T)
    offs = r.expert_off.cpu().numpy()
    assert np.diff(offs)[:len(counts)].tolist() == list(counts) and offs[32] == sum(counts)
    n = int(offs[32])
    perm = r.perm_token.cpu().numpy()[:n]
    le = np.searchsorted(offs, np.arange(n), side="right") - 1
    # every expert's first and last row and the rows on either side of its multiples of 64
    row = np.arange(n) - offs[le]
    sel = np.nonzero((row % 64 == 0) | (row % 64 == 63) | (row == np.diff(offs)[le] - 1))[0]
    act = pkg.moe.act_values(r.act[torch.as_tensor(sel, device=cuda_device)]).cpu().numpy()
    c_ref, _ = orc.expert_rows(oracle_inputs(cfg, host, w_host), perm[sel], le[sel])
    # hi + lo holds fp32 to 2^-17; the fp8 MFMA's block sums are ~1e-5 off
    bad = bf16_close(act, c_ref, atol=5e-4, rtol=1e-4)
    assert not bad.any(), f"{int(bad.sum())} elements, rows {np.unique(np.nonzero(bad)[0])[:8]}"


@pytest.mark.parametrize("T", [1023, 1024, 3001])
def test_expert_row_counts(pkg, orc, cuda_device, T):
    check_rows(pkg, orc, cuda_device, T, COUNTS)


def test_most_row_tiles(pkg, orc, cuda_device):
    """Every pick local and every expert one row past a whole 256-row tile: 64
    row tiles, one fewer than the wide kernel's grid holds for T = 1028 (a
    block takes one tile, so a shorter grid would leave rows unwritten)."""
    T, counts = 1028, (257,) * 32
    row_tiles = sum(-(-c // 256) for c in counts)
    assert sum(counts) == 8 * T and row_tiles == 64 and row_tiles + 1 == -(-8 * T // 256) + 32
    check_rows(pkg, orc, cuda_device, T, counts)
