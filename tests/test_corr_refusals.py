"""What the Correlation entry points with a workspace or a limit say when they
refuse operands (host side): the limit, not a need that no kernel has."""
import ctypes


def test_messages_name_the_limit(vsc):
    L = vsc.lib()
    L.vsc_last_error.restype = ctypes.c_char_p
    one = ctypes.c_void_p(16)
    shape = (1, 64, 600, 601)
    bytes_ = L.vsc_correlation_workspace_size(*shape, vsc.VSC_BF16)
    assert bytes_ > 32 << 20
    assert L.vsc_correlation_forward_noalloc(one, one, one, *shape, 4, 0, vsc.VSC_BF16, None, None) == vsc.VSC_E_INVALID
    said = L.vsc_last_error()
    assert b"need" not in said and str(32 << 20).encode() in said and str(bytes_).encode() in said
    assert b"vsc_correlation_forward takes any" in said
    assert L.vsc_correlation_forward_ws(one, one, one, *shape, 4, 0, vsc.VSC_BF16, None, None, 0, None) == vsc.VSC_E_INVALID
    assert b"without one" in L.vsc_last_error()
