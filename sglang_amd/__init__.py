"""MI355X-native W8A8 FP8 linear path behind SGLang's operator signatures.

Modules:
  sgl_kernel  - the ops SGLang reaches through ``sgl_kernel`` (quant, GEMMs, MoE helpers)
  fp8_kernel  - ``sglang.srt.layers.quantization.fp8_kernel`` entry points
  fp8_utils   - ``sglang.srt.layers.quantization.fp8_utils`` entry points (linear apply)
  fused_moe   - block-FP8 fused-experts pipeline
"""
import torch

from . import _lib  # noqa: F401  (fails loudly when the HIP library is not built)
from . import _host  # noqa: F401  (likewise for the native side of the layer-level calls)


def _check_host() -> None:
    if _host.torch != "built for torch %s;" % torch.__version__:
        raise ImportError("sglang_amd: _host.so was %s this is torch %s. Build it again with `python sglang_amd/csrc/build.py`."
                          % (_host.torch, torch.__version__))


_check_host()

__all__ = ["sgl_kernel", "fp8_kernel", "fp8_utils", "fused_moe"]
