"""Model.get: what is read is the tensor as the last forward left it, byte for byte, for sizes around the pieces of the small
reads' kernel and either side of the largest it takes, from addresses that are no multiple of 16, read after read and with threads
reading at once."""
import threading

import numpy as np
import pytest

from megcc_amd import abi, runtime

pytestmark = pytest.mark.gpu

LARGEST = 64 << 10


def build(nbytes):
    """y = saturate(x + x): a tensor of that many bytes, and x itself"""
    m = runtime.Model()
    x = m.tensor("x", (1, nbytes), abi.QINT8, 0.5)
    m.mark_input(x)
    y = m.tensor("y", (1, nbytes), abi.QINT8, 0.5)
    m.opr("kernel_elementwise_multitype_QADD_qsi8qsi8qsi8", [x, x], [y])
    m.mark_output(y)
    return m, x, y


def doubled(x):
    return np.clip(2 * x.astype(np.int32), -128, 127).astype(np.int8)


@pytest.mark.parametrize("nbytes", [1, 15, 16, 17, 1000, 16383, 16400, LARGEST - 1, LARGEST, LARGEST + 1])
def test_every_byte_of_every_read(nbytes):
    m, x, y = build(nbytes)
    m.finalize()
    for seed in range(4):
        value = np.random.default_rng(seed).integers(-128, 128, (1, nbytes), dtype=np.int8)
        m.set_input(x, value)
        m.forward()
        np.testing.assert_array_equal(m.get(y), doubled(value))
        np.testing.assert_array_equal(m.get(x), value)


@pytest.mark.parametrize("offset,n", [(1, 40), (8, 1000), (16, 1000), (4, 63)])
def test_a_view_at_any_byte(offset, n):
    m, x, y = build(4096)
    part = m.view("part", y, (1, n), (n, 1), offset)
    m.finalize()
    value = np.random.default_rng(offset).integers(-128, 128, (1, 4096), dtype=np.int8)
    m.set_input(x, value)
    m.forward()
    np.testing.assert_array_equal(m.get(part), doubled(value)[:, offset:offset + n])


def test_threads_that_read_at_once():
    m, x, y = build(5000)
    m.finalize()
    value = np.random.default_rng(7).integers(-128, 128, (1, 5000), dtype=np.int8)
    m.set_input(x, value)
    m.forward()
    want, wrong = doubled(value), []

    def read():
        for _ in range(50):
            if not np.array_equal(m.get(y), want):
                wrong.append(1)

    readers = [threading.Thread(target=read) for _ in range(4)]
    for t in readers:
        t.start()
    for t in readers:
        t.join()
    assert not wrong
