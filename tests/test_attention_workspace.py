"""adr_attention_f16_ws and its size query: what needs no device (the plan is then that of an MI355X)."""
import pytest

from adrastea_amd import TensorLayout, _ffi
from adrastea_amd import kernels as K


def heads_view(tokens, heads, d):
    return TensorLayout.row_major([tokens, heads * d]).shape_cast([tokens, heads, d]).permute([1, 0, 2])


def need(heads, m, n, d, mask=0):
    q, k = heads_view(m, heads, d), heads_view(n, heads, d)
    return K.attention_workspace_bytes(q, q, k, k, mask)


def test_workspace_bytes():
    assert need(32, 1, 2047, 128) == 8 * 32 * (128 * 4 + 8)   # eight parts: sums, maximum and sum of a row
    assert need(32, 2048, 2048, 128) == 0                     # query blocks enough
    assert need(32, 1, 64, 128) == 0                          # keys too few
    assert need(1, 40, 2000, 128) > 0
    # parts pay for a second launch: not where the keys of one are read in the time that takes
    assert all(need(heads, 17, n, 64) == 0 for heads in (1, 12, 16) for n in (257, 384, 500))
    assert need(2, 512, 512, 64, 1) == 0
    # nor for keys that no row sees
    assert all(need(32, m, 2000, 128, 1) == 0 for m in (40, 64, 130))
    assert need(2, 700, 2000, 64, 1) == need(2, 700, 700, 64, 1) > 0


@pytest.mark.parametrize("bad,code", [(dict(d=96), _ffi.ADR_EUNSUPPORTED_LAYOUT), (dict(n=-1), _ffi.ADR_EINVAL_SHAPE),
                                      (dict(mask=2), _ffi.ADR_EINVAL_ENUM), (dict(sx=2), _ffi.ADR_EUNSUPPORTED_LAYOUT),
                                      (dict(sy=-8), _ffi.ADR_EUNSUPPORTED_LAYOUT), (dict(sy=4), _ffi.ADR_EUNSUPPORTED_LAYOUT),
                                      (dict(n=0), _ffi.ADR_EINVAL_SHAPE), (dict(m=0, n=0), 0)])
def test_codes(bad, code):
    a = dict(heads=4, m=1, n=2048, d=128, sx=1, sy=512, mask=0)
    a.update(bad)
    strides = [a["sx"], a["sy"], 128] * 4
    lib = _ffi.lib()
    assert lib.adr_attention_f16_workspace_bytes(a["heads"], a["m"], a["n"], a["d"], *strides, a["mask"]) == code
    args = [None, 64, 64, 64, 64, a["heads"], a["m"], a["n"], a["d"], *strides, 0.1, 1.0, a["mask"]]
    assert lib.adr_attention_f16_ws(*args, None, 0) == code   # (refused, or nothing to do, before any launch)
    assert lib.adr_attention_f16(*args) == code


def test_workspace_argument_is_checked():
    args = [None, 64, 64, 64, 64, 4, 1, 2048, 128, *([1, 512, 128] * 4), 0.1, 1.0, 0]
    lib = _ffi.lib()
    assert lib.adr_attention_f16_ws(*args, None, 64) == _ffi.ADR_ENULL
    assert lib.adr_attention_f16_ws(*args, 64, -1) == _ffi.ADR_ENULL
    assert lib.adr_attention_f16_ws(*args, 72, 1 << 20) == _ffi.ADR_EINVAL_SHAPE


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("heads,m", [(2**31 - 1, 2**31 - 1), (2**31 - 1, 1), (2**20, 2**31 - 1), (2**24, 128)])
def test_more_rows_than_parts_are_counted_for(heads, m, d):
    """Query rows by the thousands of millions (rows may overlap): the keys are not shared, and no count of
    rows, parts and bytes runs over on the way to saying so."""
    strides = [1, d, 0] * 4
    assert _ffi.lib().adr_attention_f16_workspace_bytes(heads, m, 4096, d, *strides, 0) == 0
