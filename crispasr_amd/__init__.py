"""MI355X-native attention hot path of CrispASR's ggml graphs (GGML_OP_FLASH_ATTN_EXT).

The product is ``libmi355x_fattn.so`` (hand-written HIP for gfx950 behind a C ABI, see
``include/mi355x_fattn.h``).  This package is the thin host side the tests and the
benchmark drive it through: ``ggml`` mirrors the reference's operator interface for this
path (``ggml_flash_attn_ext``, ``ggml_cpy``, ``ggml_set_rows`` on strided tensor views).
"""
import importlib

_FROM_GGML = ("F16", "F32", "Q4_0", "Q4_1", "Q5_0", "Q5_1", "Q8_0", "HostBuffer", "Tensor", "cpy", "flash_attn_ext", "set_rows")

__all__ = ["ggml", "Tensor", "HostBuffer", "F32", "F16", "Q8_0", "Q4_0", "Q4_1", "Q5_0", "Q5_1", "flash_attn_ext", "cpy", "set_rows"]


def __getattr__(name):
    # on first use: the package's build module has to be importable before there is anything to load
    if name != "ggml" and name not in _FROM_GGML:
        raise AttributeError(f"module {__name__!r} has no attribute {name!r}")
    ggml = importlib.import_module(".ggml", __name__)
    globals().update({n: getattr(ggml, n) for n in _FROM_GGML}, ggml=ggml)
    return globals()[name]
