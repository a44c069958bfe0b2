"""The memory that a mirror reports: everything it holds, the packed columns of
the products among it."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt", ["CSR", "COO", "SCOO"])
@pytest.mark.parametrize("dtype,entry", [("f64", 8 + 4 + 3), ("f32", 4 + 4 + 3), ("bf16", 2 + 4 + 3)])
def test_mirror_bytes(tb, gpu, fmt, dtype, entry):
    n, c = 20000, 12
    info = tb.FORMATS[fmt]().fill_cqmat(n, n, c, 0.3, 5, value_seed=5).mirror_info(dtype)
    e = info["entries"]
    # a value, a column and a packed column an entry, a row pointer a row (and a row number in COO and SCOO); at most a
    # tile boundary for 1024 entries and 512 bytes of padding an array beside them
    rows = 4 * info["rows"] * (1 if fmt == "CSR" else 2)
    assert entry * e + rows <= info["mirror_bytes"] <= entry * e + rows + 4 * (e // 1024 + 2) + 8 * 768
