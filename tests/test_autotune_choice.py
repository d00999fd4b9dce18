"""What the tuners choose from their timings (no GPU: the timings are given)."""
from gonzales_amd.autotune import CANDIDATES, MIS_CANDIDATES, MisLaunch, fastest
from gonzales_amd.batch import BATCH_CANDIDATES


def test_the_default_is_the_first_candidate_and_no_launch_is_listed_twice():
    for c in (CANDIDATES, MIS_CANDIDATES, BATCH_CANDIDATES):
        assert c[0].by_size == 1 and not any(x.by_size for x in c[1:]) and len(set(c)) == len(c)
    # the kernels of queued 1 and the batch's bounce kernel run one wave a workgroup: block and grid_scale change nothing
    for c in (MIS_CANDIDATES, BATCH_CANDIDATES):
        keys = [(x.chunk, x.drain_level) for x in c[1:] if x.queued == 1]
        assert len(set(keys)) == len(keys)


def test_the_default_stays_unless_another_is_faster_than_the_noise():
    default, other = MisLaunch(1, 256, 1, 256, 3, by_size=1), MisLaunch(3, 256, 1, 64, 3)
    assert fastest({default: 1.0, other: 0.995}) == default
    assert fastest({default: 1.0, other: 0.98}) == other
    assert fastest({default: 0.104, other: 0.1}) == default and fastest({default: 0.107, other: 0.1}) == other
    assert fastest({other: 1.0, MisLaunch(): 0.999}) == MisLaunch()  # no default among the candidates
