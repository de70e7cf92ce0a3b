"""Host calls whose operands are less than 64 MiB: gathered by several threads in page-locked memory, in slices where the program
only maps over its leading index, copied out while the rest is under way."""
import os
import subprocess
import sys
import threading
from pathlib import Path

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _data(shape, seed):
    return np.random.default_rng(seed).uniform(-1, 1, shape).astype(np.float32)


# bytes in all: a few hundred, one piece, around the pieces of 1, 2 and 4 MiB, where slices begin (6 MiB), just below 64 MiB
@pytest.mark.parametrize("rows, cols", [(1, 1), (3, 5), (64, 1000), (300, 1001), (513, 1021), (700, 1500), (1023, 1025), (1500, 2100), (7, 700001), (2, 3000000),
                                        (5000, 1117)])
def test_elements_arrive_where_they_belong(rows, cols):
    from i_amd import Component as i

    a, b = _data((rows, cols), 1), _data((rows, cols), 2)
    total = 3 * 4 * rows * cols
    component = i("ij+ij~ij")
    for _ in range(2):
        assert np.array_equal(component.exec_numpy(a, b), a + b)
    moved_in_slices = rows >= 2 and total >= 6 << 20
    assert ("host: operands in" in component.report()) == moved_in_slices, component.report()
    out = np.full((rows, cols), np.nan, np.float32)
    component.into(out, b, a)
    assert np.array_equal(out, a + b)
    # an operand that every slice needs whole, and a program that cannot be cut: the same pieces in one go
    bias = _data((cols,), 3)
    assert np.array_equal(i("ij+j~ij||ij").exec_numpy(a, bias), a + bias)
    if total < 40 << 20:
        flipped = i("ij~ji")
        assert np.array_equal(flipped.exec_numpy(a), a.T)
        assert "host:" not in flipped.report()



# several outputs: small neighbours that cross together, with an empty one between them, up to pieces of their own
@pytest.mark.parametrize("rows, cols", [(1, 1), (3, 5), (63, 65), (0, 4), (300, 1001), (525, 999), (1100, 1000), (9, 150001)])
def test_several_outputs_arrive_where_they_belong(rows, cols):
    from i_amd import Component as i

    a, b = _data((rows, cols), 1), _data((rows, cols), 2)
    component = ((i("ij+ij~ij") & i("ij~ji")) & i("-ij~ij")) & i("ij~ji")
    shapes = [(rows, cols), (cols, rows), (rows, cols), (cols, rows)]
    expected = [a + b, a.T, -a, a.T]
    for _ in range(2):
        rings = [np.full(rows * cols + 32, np.nan, np.float32) for _ in shapes]
        outs = [ring[16:16 + rows * cols].reshape(shape) for ring, shape in zip(rings, shapes)]
        component.into(outs, a, b)
        for out, want, ring in zip(outs, expected, rings):
            assert np.array_equal(out, want)
            assert np.isnan(ring[:16]).all() and np.isnan(ring[-16:]).all()


OVERLAPPING = """
import sys
import numpy as np
from i_amd import Component as i
rows, cols = int(sys.argv[1]), 2000
for shift in (0, 1000, -1000, rows // 2 * cols, rows // 3 * 2 * cols, 100 * cols, -100 * cols, -(rows // 3 * 2) * cols):
    memory = np.random.default_rng(5).uniform(-1, 1, 3 * rows * cols).astype(np.float32)
    a = memory[rows * cols:][:rows * cols].reshape(rows, cols)
    out = memory[rows * cols + shift:][:rows * cols].reshape(rows, cols)
    expected = a + a
    component = i("ij+ij~ij")
    component.into(out, a, a)
    assert np.array_equal(out, expected), shift
    # (in place, a slice overwrites what it has read)
    assert ("host: operands in" in component.report()) == (shift == 0), (shift, component.report())
    # rows of the result shorter than those of the operand
    a = memory[rows * cols:][:rows * cols].reshape(rows, cols)
    expected = a[:, 0].copy()
    out = a.reshape(-1)[:rows] if shift == 0 else memory[rows * cols + abs(shift):][:rows]
    a[:, 1:] = 0.0
    i("+ij~i").into(out, a)
    assert np.array_equal(out, expected), shift
"""


# outputs in memory that an input has too: the input itself, and rows before and behind it, for calls through the mirror (62 MB)
# and larger ones.  (With one thread that copies, every row is gathered as late as it can be.)
@pytest.mark.parametrize("rows", [2600, 9000])
@pytest.mark.parametrize("threads", ["1", "8"])
def test_outputs_over_inputs(threads, rows):
    done = subprocess.run([sys.executable, "-c", OVERLAPPING, str(rows)], env={**os.environ, "ILANG_HIP_COPY_THREADS": threads}, cwd=Path(__file__).parents[1],
                          capture_output=True, text=True, timeout=100)
    assert done.returncode == 0, done.stderr[-1500:]


def test_products_and_reductions():
    from i_amd import Component as i

    mm_t = i("ik*jk~ijk | i:16,j:16 | jii'j'k") >> i("+ijk~ij | i:16,j:16 | jii'j'k0")
    for m, n, k in ((700, 900, 1100), (2300, 1200, 900), (33, 2000, 2000)):
        a, b = _data((m, k), m), _data((n, k), n)
        ref = a.astype(np.float64) @ b.astype(np.float64).T
        # (f32 sums of k products in some order: a rounding per term, and one per product)
        bound = (k + 8) * 2.0 ** -24 * (np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64).T)
        assert (np.abs(mm_t.exec_numpy(a, b) - ref) <= bound).all(), (m, n, k, mm_t.report())
    x = _data((3000, 1111), 4)
    assert np.allclose(i("+ij~j").exec_numpy(x), x.astype(np.float64).sum(0), atol=3000 * 2.0 ** -24 * 3000)


def test_calls_of_several_threads_at_once():
    """One call has the kept block and its mirror, the others allocate their own; all use the same copying threads."""
    from i_amd import Component as i

    wrong = []

    def work(seed):
        component = i("ij+ij~ij")
        for n in range(6):
            a, b = _data((600 + 7 * seed, 1200 + n), seed), _data((600 + 7 * seed, 1200 + n), seed + 50)
            if not np.array_equal(component.exec_numpy(a, b), a + b):
                wrong.append((seed, n))

    threads = [threading.Thread(target=work, args=(seed,)) for seed in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
