"""The sampler's row layout at its edges (tiles of 8192 entries, rows of up to
32768 entries in LDS, rows that are not 16-byte aligned), against the oracle as
test_gpu_sampling does, and rows of tied or infinite logits, whose filters are
exact: equal probabilities 1 / 2^n sum without rounding."""
import numpy as np
import pytest

import oracle as orc
import orion_hip as oh
from test_gpu_sampling import kept, run, test_rows_match_the_oracle as rows_match_the_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V", [1, 9, 8191, 8193, 16385, 32768, 32769, 40003])
def test_rows_at_tile_edges_match_the_oracle(backend, V):
    rows_match_the_oracle(backend, V)


@pytest.mark.parametrize("V", [16, 8192, 16384, 65536])
def test_tied_and_infinite_rows(backend, V):
    tied = np.full(V, 1.5, np.float32)
    some = np.full(V, -np.inf, np.float32)
    some[::2] = 0.25
    rows = [tied, tied, some, some, tied]
    params = [oh.SamplingParams(top_p=0.5), oh.SamplingParams(top_k=3),
              oh.SamplingParams(top_p=0.25), oh.SamplingParams(temperature=0.0),
              oh.SamplingParams(temperature=0.5, top_k=V // 2, top_p=0.125)]
    uniforms = [0.3, 0.6, 0.9, 0.1, 0.5]
    tokens, filtered = run(backend, rows, params, None, uniforms)
    for i, p in enumerate(params):
        want, wx, margin = orc.sample(rows[i], [], p.temperature, p.top_k, p.top_p, 1.0,
                                      uniforms[i])
        assert kept(filtered[i]) == kept(wx), i
        if p.temperature == 0.0 or margin > 1e-5:
            assert tokens[i] == want, i
