"""The operand descriptors of acestep_ops.ops.desc, field by field, on stand-ins for
device memory: sliced, permuted, negatively strided, empty and Q8_0 views, and the
bounds and type errors."""
import pytest

from acestep_ops import ops
from acestep_ops._lib import BF16, F32, Q8_0
from acestep_ops.device import DTensor


class Mem:
    ptr, nbytes = 1 << 20, 4096


def fields(t):
    d = ops.desc(t)
    return d.data, d.type, d.reserved, list(d.ne), [v - (1 << 64) if v >> 63 else v for v in d.nb]


def test_fields():
    x = DTensor(Mem(), (2, 3, 8), "f32")
    assert fields(x) == (1 << 20, F32, 0, [8, 3, 2, 1], [4, 32, 96, 192])
    assert fields(x[:, 1:, 2:6].permute(1, 0, 2)) == ((1 << 20) + 40, F32, 0, [4, 2, 2, 1], [4, 96, 32, 64])
    assert fields(DTensor(Mem(), (4,), "bf16", (-1,), 64)) == ((1 << 20) + 64, BF16, 0, [4, 1, 1, 1], [-2, -8, -8, -8])
    assert fields(DTensor(Mem(), (), "f32")) == (1 << 20, F32, 0, [1, 1, 1, 1], [4, 4, 4, 4])
    assert fields(DTensor(Mem(), (0, 5), "f32", None, 4096))[3] == [5, 0, 1, 1]
    q = ops.Q8(DTensor(Mem(), (3, 68), "u8"))
    assert fields(q) == (1 << 20, Q8_0, 0, [64, 3, 1, 1], [34, 68, 204, 204])
    assert fields(ops.Q8(DTensor(Mem(), (34,), "u8")))[4] == [34, 34, 34, 34]


@pytest.mark.parametrize("t", [DTensor(Mem(), (1025,), "f32"), DTensor(Mem(), (2,), "f32", (-1,), 0),
                               DTensor(Mem(), (2,), "f32", None, 4092), DTensor(Mem(), (1,) * 5, "f32"),
                               ops.Q8(DTensor(Mem(), (2, 35), "u8")), ops.Q8(DTensor(Mem(), (2, 34), "u8", (68, 2)))])
def test_refused(t):
    with pytest.raises(ValueError):
        ops.desc(t)


def test_dtype_refused():
    with pytest.raises(TypeError):
        ops.desc(DTensor(Mem(), (4,), "u8"))
