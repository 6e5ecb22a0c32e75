"""Device memory that a context holds after its tables are built (GPU): for more reads than one group
of the build takes, signatures, values, buckets and order, and not the build's workspace."""
import numpy as np
import pytest
import torch

from rabbitqcplus_amd import engine, reads

pytestmark = pytest.mark.gpu


def test_workspace_of_a_large_map_is_given_back():
    n = 17_000_000                                       # above 2^24
    rng = np.random.default_rng(91)
    enc = rng.integers(0, 1 << 32, (n, 2), dtype=np.uint32)
    rs = reads.ReadStorage(enc, np.full(n, 32, np.int32), None, np.zeros(n, np.uint8), False)
    eng = engine.CareEngine(0, kmerlength=16, num_hash_maps=1)
    eng.set_reads(rs)
    free = torch.cuda.mem_get_info()[0]
    eng.build_tables()
    held = free - torch.cuda.mem_get_info()[0]
    eng.close()
    # 8 + 4 + 8 + 4 bytes per read and map, 2 of its seed; the workspace is 40 more. Two hashed 16-mers of random
    # reads seldom meet: slots take less than the slack
    print(f"[reads={n}] held {held / n:.1f} bytes per read", flush=True)
    assert held <= 26 * n + (128 << 20)
