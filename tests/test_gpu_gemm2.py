"""GEMM2 rows and layer output where the row count of an expert picks the tile
(at most 16, at most 32, more rows), against the CPU oracle: experts are given
exact row counts through hand-made logits."""
import numpy as np
import pytest
import torch

from test_gpu_layer import check_layer
from util import bf16_close, gpu_tokens, gpu_weights, oracle_inputs

pytestmark = pytest.mark.gpu


def tokens_with_rows(pkg, cfg, device, T, counts):
    """Inputs whose local experts 0 .. len(counts) - 1 (window 0, group 0)
    take counts[e] tokens.  Eight experts of groups 1-3 stand between the
    chosen local ones and all others, so a token's remaining picks fall there."""
    tok, host = gpu_tokens(pkg, cfg, device, T)
    rng = np.random.default_rng(T)
    logits = rng.uniform(-6.0, -4.0, (T, 256)).astype(np.float32)
    for g in (1, 2, 3):
        logits[:, 32 * g:32 * g + 8] += 6.0
    load = np.zeros(T, np.int64)
    for e, n in sorted(enumerate(counts), key=lambda c: -c[1]):  # each expert's tokens: those with the fewest picks
        pick = np.lexsort((rng.random(T), load))[:n]
        load[pick] += 1
        logits[pick, e] = rng.uniform(3.0, 4.0, n)
    assert load.max() <= 8
    logits_d = torch.from_numpy(logits).to(device)
    bias = torch.zeros(256, dtype=torch.bfloat16, device=device)
    tok = (logits_d, bias, tok[2], tok[3])
    return tok, (logits, np.zeros(256, np.uint16), host[2], host[3])


# (T, rows per expert, tokens and rows checked: None = all)
ROW_CASES = [
    (9, (9, 1, 8), None),                # smallest T with GEMM2 rows and a combine pass
    (16, (16, 15, 1, 16, 9), None),
    (17, (17, 16, 1), None),
    (64, (64, 33, 32, 17, 16, 1), None),
    (65, (1, 15, 16, 17, 31, 32, 33, 48, 64, 65), None),
    (130, (16, 1, 130, 32, 2, 128, 64, 33), None),
    (700, (32,) * 20 + (16,) * 8 + (31, 17, 8, 1), None),
    (3072, (32, 16, 200, 33, 5), 128),   # largest T with tiles of their own for at most 32 rows
    (3073, (32, 16, 200, 33, 5), 128),
]


@pytest.mark.parametrize("T,counts,n_check", ROW_CASES)
def test_expert_row_counts(pkg, orc, cuda_device, T, counts, n_check):
    cfg = pkg.synth.CONFIGS["prefill_t1024"]
    w, w_host = gpu_weights(pkg, cfg.seed, cuda_device)
    tok, host = tokens_with_rows(pkg, cfg, cuda_device, T, counts)
    print(f"row counts T={T} {counts}", flush=True)
    check_layer(pkg, orc, cuda_device, cfg, 0, tok, host, w, w_host, n_check)
    r = pkg.intermediates(pkg.workspace(cuda_device, T), T)
    offs = r.expert_off.cpu().numpy()
    assert np.diff(offs)[:len(counts)].tolist() == list(counts) and offs[32] == sum(counts)
    n = int(offs[32])
    perm = r.perm_token.cpu().numpy()[:n]
    le = np.searchsorted(offs, np.arange(n), side="right") - 1
    edges = np.concatenate([[offs[e], offs[e + 1] - 1] for e in range(len(counts))])
    sel = np.unique(np.concatenate([edges, np.arange(0, n, 1 if n <= 600 else 5)]))
    down = r.down[torch.as_tensor(sel, device=cuda_device)].cpu().numpy()
    _, o_ref = orc.expert_rows(oracle_inputs(cfg, host, w_host), perm[sel], le[sel])
    # fp32 rows of the activation pair: hi + lo holds it to 2^-17, the fp8 MFMA
    # in front of it to ~1e-5 of its terms
    bad = bf16_close(down, o_ref, atol=1e-4, rtol=1e-4)
    assert not bad.any(), f"{int(bad.sum())} elements, rows {np.unique(np.nonzero(bad)[0])[:8]}"
