"""Stage markers of the event path (the reference's no-op `cuda_stage`,
spike_mamba/runtime_breakdown.py:13-15). Here each stage is a
torch.profiler.record_function range while a torch profiler runs (which shows
it next to the HIP kernels it launches), and nothing otherwise: a range costs
about 10 us of host time whether or not anyone records it."""
import torch
from torch.autograd import profiler as _profiler

__all__ = ["cuda_stage"]


class _NoStage:
    __slots__ = ()

    def __enter__(self):
        return self

    def __exit__(self, *exc):
        return False


_NO_STAGE = _NoStage()


def cuda_stage(name):
    if _profiler._is_profiler_enabled:
        return torch.profiler.record_function(name)
    return _NO_STAGE
