"""The sampler's top-k threshold where a radix bucket's keys are ranked in LDS:
buckets of one key to one more than the block holds, and equal keys across
the threshold, against the oracle."""
import numpy as np
import pytest

import oracle_lib as O
import spec
from test_gpu_sample import Sampler

pytestmark = pytest.mark.gpu
ONE = spec.ONE


@pytest.mark.parametrize("bucket", [1, 2, 64, 1023, 1024, 1025, 2000])
@pytest.mark.parametrize("ties", [False, True])
def test_topk_bucket_sizes_vs_oracle(ctx, bucket, ties):
    """`bucket` of 5000 logits share their top byte (below 40 larger ones):
    distinct in the low bits, or in runs of equal values."""
    n = 5000
    rng = np.random.default_rng(bucket + ties)
    x = rng.integers(-40 * ONE, -30 * ONE, size=n, dtype=np.int64)
    where = rng.permutation(n)
    low = rng.integers(0, 7 if ties else 1 << 40, size=bucket, dtype=np.int64)
    x[where[:bucket]] = 4 * ONE + low * ((1 << 38) if ties else 1)
    x[where[bucket:bucket + 40]] = rng.integers(8 * ONE, 9 * ONE, size=40, dtype=np.int64)
    s = Sampler(ctx, n)
    try:
        for k in sorted({41, 40 + (bucket + 1) // 2, 40 + bucket}):
            for p in (ONE, ONE * 9 // 10):
                st = O.rng_seed(1000 * bucket + k)
                print("[case] top-k", bucket, "ties", ties, "k", k, flush=True)
                # a high temperature, so that draws reach the threshold's values
                want = O.sample(x, 30 * ONE, k, p, st)
                assert s(x, 30 * ONE, k, p, st) == want, (bucket, k, p)
    finally:
        s.free()
