"""What the decode path refuses on the host, before any kernel is launched."""
import types

import pytest
import torch

from openattention_amd.method import OursHIP


def test_rows_step_refuses_keys_past_the_cache():
    """A multi-row call over more keys than the index or the cache holds, or over a cache of another
    shape, is refused on the host (the kernels read positions up to n_keys - 1 unchecked)."""
    B, Lmax, Q = 1, 512, 4
    m = OursHIP(types.SimpleNamespace(rho=0.01), B, Lmax, "cpu", n_layers=1)
    q = torch.zeros(B, 32, Q, 128, dtype=torch.bfloat16)
    out = torch.empty_like(q)
    n_dev = torch.zeros(1, dtype=torch.int32)

    def rows(kv, n_keys, v=None):
        K = torch.zeros(kv, dtype=torch.bfloat16)
        return m.rows_step(m.st[0], K, K if v is None else torch.zeros(v, dtype=torch.bfloat16), q, n_dev, n_keys, out)

    for args in (((8, Lmax + 64, 128), Lmax + 1), ((8, 300, 128), 301), ((4, Lmax, 128), 300),
                 ((8, Lmax, 128), 300, (8, Lmax - 1, 128)), ((8, Lmax, 128), 0)):
        with pytest.raises(ValueError, match="n_keys|K, V"):
            rows(*args)
    assert int(n_dev) == 0
