"""run_stream (resolve2d_amd/serve.py) where scenes arrive faster than they are
built: the running lanes are still collected and launched between the builds."""
import time

from resolve2d_amd import serve


class _Server:
    """Counts calls; a request is done two ticks after its submission."""

    def __init__(self):
        self.log, self.at, self.done = [], {}, []

    def submit(self, world, steps):
        self.log.append("submit")
        self.at[world] = len([e for e in self.log if e == "tick"])
        return world

    def tick(self):
        self.log.append("tick")
        n = self.log.count("tick")
        self.done = [w for w, k in self.at.items() if n - k >= 2]
        for w in self.done:
            del self.at[w]
        return {"completed": len(self.done)}

    def completed(self):
        return self.done

    def poll(self, ticket):
        return {"total_ms": 1.0}

    def stats(self):
        return {"body_steps": 0}


def test_ticks_between_builds():
    def build(k):
        time.sleep(serve.BUILD_SLICE_S)
        return k

    sv, seen = _Server(), []
    r = serve.run_stream(sv, [(0.0, k) for k in range(12)], build, 1, on_done=lambda p, w, st: seen.append(p))
    assert r["submitted"] == 12 and sorted(seen) == list(range(12))
    runs = "".join(e[0] for e in sv.log).split("t")
    assert max(map(len, runs)) <= 2          # no more than two builds without a tick

