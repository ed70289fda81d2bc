"""fo_attn_bias_rows rejects bad arguments before any launch (no GPU needed); its results: test_attention_tile_bias_gpu.py."""
import ctypes

from fast_ops_amd import _lib

I3 = ctypes.c_int64 * 3


def test_argument_validation_without_device():
    call = lambda bias=0x1000, st=I3(0, 9, 3), elt=2, B=1, H=2, Sq=3, Sk=3, out=0x2000, row=8: _lib.load().fo_attn_bias_rows(
        bias, st, elt, B, H, Sq, Sk, out, row, None)
    assert call(bias=None) == -1 and call(st=None) == -1 and call(out=None) == -1
    assert call(elt=8) == -2
    assert call(Sk=0) == -4 and call(row=2) == -4 and call(B=1 << 20, H=1 << 20) == -4
    assert call(st=I3(0, -9, 3)) == -5 and call(row=12) == -5
    assert call(bias=0x1001) == -6 and call(out=0x2008) == -6 and call(bias=0x1002, elt=4) == -6
