"""Times of calls against each other, for tests of what a call may cost."""
import time


def ratio(torch, a, b, calls, limit, repeats=10):
    """The time of a() over that of b(), each the least of `repeats` blocks of
    `calls` calls, in turn.  Measured up to three times until it is below
    `limit`: noise only adds."""
    least = float("inf")
    for _ in range(3):
        best = [float("inf")] * 2
        for _ in range(repeats):
            for q, fn in enumerate((a, b)):
                fn()
                torch.cuda.synchronize()
                t = time.perf_counter()
                for _ in range(calls):
                    fn()
                torch.cuda.synchronize()
                best[q] = min(best[q], time.perf_counter() - t)
        least = min(least, best[0] / best[1])
        if least < limit:
            break
    return least
