"""Times of launches on the GPU, for tests of one form against another."""
import torch


def median_us(launch, launches=10, repeats=21):
    """Median over `repeats` of the time of one of `launches` launches in a row, queued behind other work so that the host is ahead of them."""
    ahead = torch.empty(1 << 29, dtype=torch.uint8, device="cuda")
    times = []
    for _ in range(repeats):
        for _ in range(10):                                   # (about 0.1 ms each)
            ahead.fill_(0)
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(launches):
            launch()
        b.record()
        b.synchronize()
        times.append(a.elapsed_time(b) / launches * 1e3)
    return sorted(times)[repeats // 2]
