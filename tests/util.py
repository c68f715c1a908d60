"""The counter-based generator and the device-buffer helpers live in the package (the benchmark uses them too)."""
from sofie_amd.benchsupport import synthetic as _synthetic
from sofie_amd.benchsupport.synthetic import *  # noqa: F401,F403
from sofie_amd.benchsupport.synthetic import splitmix64, uniform01, normal, int8_sym, int32_range, to_dev, ptr, to_host  # noqa: F401


def dev_empty(shape, dtype):
    """A device buffer that holds 0x5a in every byte (1.5e16 as fp32, 1515870810 as int32): the allocator likes to hand out the block in which the last test left its correct results, and
    what a kernel fails to store must not be found there."""
    import torch
    t = _synthetic.dev_empty(shape, dtype)
    if t.numel():
        t.view(-1).view(torch.uint8).fill_(0x5a)
        torch.cuda.synchronize()   # the library's streams do not wait for torch's
    return t
