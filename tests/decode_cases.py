"""Decode batches of a small bf16-KV model at serving contexts, for the tests of
the decode route: rows of their own blocks, contexts up to `longest`."""
import numpy as np

from model_fixtures import Spec


def decode_case(rows, d, longest):
    """(spec, contexts, block tables): the contexts include the longest, the
    block and 16-token edges below it, and some in between."""
    rng = np.random.default_rng(rows * 1000 + longest)
    edges = [longest, longest - 1, longest // 2 + 1, 33, 17, 16, 2]
    ctxs = (edges + rng.integers(longest // 4, longest, rows).tolist())[:rows]
    need = [(c + 15) // 16 for c in ctxs]
    spec = Spec(2, 128, 8, 2, d, 160, 300, max_pos=2048, num_blocks=sum(need) + 3, block_size=16)
    ids = rng.permutation(spec.num_blocks).tolist()
    return spec, [int(c) for c in ctxs], [[int(ids.pop()) for _ in range(n)] for n in need]
