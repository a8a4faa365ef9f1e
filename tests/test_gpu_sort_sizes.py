"""The radix sort under the block partition at the edges of its dispatch: one, two
and three passes, digits of 8, 9 and 10 bits, chunk remainders, and both chunk
sizes (2048 keys below 4 Mi particles, 4096 from there).  Whole numbers: the
partition equals the oracle's bit for bit."""
import numpy as np
import pytest
import torch

import tesserae_hip as th


@pytest.mark.gpu
@pytest.mark.parametrize("cells,bits,sizes", [
    ((5, 5), 8, (1, 63, 2047, 2048, 2049)),             # 5 x 5 blocks: 100 keys
    ((100, 100), 8, (2049, 50_001)),                    # 16-bit keys, two 8-bit digits
    ((254, 254), 9, (50_001,)),                         # 18-bit keys: two 9-bit digits
    ((500, 500), 10, (50_001, (4 << 20) - 1, (4 << 20) + 4097)),  # 20-bit keys
    ((1000, 1000), 8, (50_001,)),                       # 22-bit keys: three 8-bit digits
    ((5000, 5000), 9, (50_001,)),                       # 27-bit keys: three 9-bit digits
    ((8200, 9000), 10, (50_001,)),                      # 29-bit keys: three 10-bit digits
])
def test_partition_over_sort_shapes(oracle, cells, bits, sizes):
    mesh = th.CartesianMesh(1.0, (0.0, float(cells[0])), (0.0, float(cells[1])), dtype=torch.float64, block_size_log2=0)
    rng = np.random.default_rng(cells[0] + bits)
    part = th.Partition(mesh)
    for n in sizes:
        print(f"[sort sizes] cells={cells} n={n}", flush=True)
        x = rng.uniform(-0.02, 1.02, size=(n, 2)) * np.array(cells)
        x[n // 2:] = x[: n - n // 2]  # equal keys: their order is the input's
        pidx, starts, stops, na = oracle.partition(mesh, x, dtype=np.float64)
        th.update(part, torch.from_numpy(x).cuda())
        assert part.nassigned == na
        np.testing.assert_array_equal(part.particleindices[:na].cpu().numpy(), pidx[:na])
        np.testing.assert_array_equal(part.starts.cpu().numpy(), starts)
        np.testing.assert_array_equal(part.stops.cpu().numpy(), stops)
