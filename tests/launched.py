"""Names of the kernels that a call launches."""
import torch


def kernels(call):
    call()                                       # (libraries are loaded and memory is there)
    torch.cuda.synchronize()
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA], acc_events=True) as p:
        call()
        torch.cuda.synchronize()
    return [e.name for e in p.events() if e.device_type == torch.autograd.DeviceType.CUDA]
