"""Whose coordinate tables the device holds: not the previous set's any more once another
set's are being written, so that a render that fails half-way through its upload cannot
leave the previous set its tables' name."""
import ctypes as C
import os

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "newman_amd", "libnm_index_check.so")


def test_tables_have_no_owner_while_they_are_written():
    if not os.path.exists(LIB):
        from newman_amd import build
        build.build_index_check()
    f = C.CDLL(LIB).nm_table_key_check
    f.restype = C.c_longlong
    assert f() == 0


def test_the_engine_gives_them_up_before_the_first_write():
    """Both paths drop the owner before make_tables and the mask copy, and name the new
    one only after the last of them."""
    src = open(os.path.join(os.path.dirname(LIB), "csrc", "kernels.hip")).read()
    for path in ("int render_hw(", "int render_sa("):
        body = src[src.index(path):]
        body = body[:body.index("\n  }\n")]
        drop, write, name = body.index("tab_key.writing()"), body.index("make_tables("), body.index("tab_key.written(")
        copies = [k for k in range(len(body)) if body.startswith("hipMemcpyAsync(d_", k) and k < name]
        assert drop < write < name and all(drop < k for k in copies)
        assert "grow(&d_frames" not in body and "grow(&d_tabs" not in body and "grow(&d_mask" not in body
