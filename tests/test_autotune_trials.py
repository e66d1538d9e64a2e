"""What the autotuner times (recorded calls of the host code, no GPU): the
launches of a long run, graphs instantiated beforehand."""
import pytest

import hip_record


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    return hip_record.build(tmp_path_factory.mktemp("hip"))


# 10: the default; 60: a run of that many steps reaches the graphs by itself
@pytest.mark.parametrize("trial_steps", [1, 5, 10, 60])
@pytest.mark.parametrize("dim,scheme", [(2, "usl"), (3, "musl")])
def test_trials_run_the_launches_of_a_run(lib, trial_steps, dim, scheme):
    out = hip_record.run(lib, """
trial, dim, scheme = %d, %d, %r
s = solver(dim, scheme, 512)
s.autotune(1e-6, trial_steps=trial)
calls = log()
# the timed steps: from the last record of the first event to the second's
events = [i for i, l in enumerate(calls) if l.startswith("event")]
ends = [i for i in events if calls[i] != calls[events[0]]]
begins = [max(j for j in events if j < i) for i in ends]
s.set_sort_interval(4)
s.step(400, 1e-6)   # instantiated by then
log()
trials = 0
for se, a, b in zip([4, 8, 16] * 3, begins, ends):
    timed = calls[a + 1:b]
    made = [l for l in timed if l.startswith(("begin", "captured", "instantiate", "malloc"))]
    assert not made, (se, made[:3])
    # the same number of graphs and kernels as that many steps of a long run
    # that begin with a sort
    s.set_sort_interval(se)
    s.step(3 * 16, 1e-6)
    log()
    while True:         # to the end of an interval
        s.step(1, 1e-6)
        if any("k_rs_hist" in l for l in log()):
            s.step(se - 1, 1e-6)
            log()
            break
    s.step(trial, 1e-6)
    run = log()
    count = lambda c: (c.count("graph"), len([l for l in c if l.startswith("launch")]))
    assert count(timed) == count(run), (se, count(timed), count(run))
    trials += 1
assert trials == 9
print("ok")
""" % (trial_steps, dim, scheme))
    assert "ok" in out
