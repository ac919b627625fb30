"""The tuning that a batch without a set one reports stands for its own choice of
groups and launch options: set back unchanged, the batch launches what it launched
before; so does the tuning that the autotuner returns."""
import pytest

pytestmark = pytest.mark.gpu

SIZES = {"f32": [(101, 99, 97), (153, 150, 149), (97, 88, 90)],
         "f64": [(84, 81, 80), (90, 70, 60), (17, 5, 9)],
         "f16s": [(130, 120, 125), (130, 110, 120), (140, 150, 130)]}


def batch(precision, sizes):
    from cavityflow_cuda_amd.batch import CavityBatch, CavitySpec
    params = dict(inv_tau=1.3, velocity_dimless=(0.07, 0.0, 0.0),
                  acceleration_dimless=(0.0, 0.0, 0.0))
    return CavityBatch([CavitySpec(z, 0.07, 150.0, params) for z in sizes], precision)


def of_a_run(b, st):
    from cavityflow_cuda_amd._lib import check, lib
    from launches import launches
    return launches(lambda h: check(lib().lbm_batch_launch(b._h, 0, 4, h)), st)


@pytest.mark.parametrize("precision", sorted(SIZES))
def test_reported_tuning_set_back_keeps_the_launches(hip, precision):
    from hiprt import stream_create, stream_destroy
    print("[case] batch untuned", precision, flush=True)
    b, st = batch(precision, SIZES[precision]), stream_create()
    untuned = of_a_run(b, st)
    reported = b.tuning()
    b.set_tuning(**reported)
    assert of_a_run(b, st) == untuned
    b.set_tuning(block=512, cells_per_thread=2, options=(0, 0))
    one = of_a_run(b, st)
    assert len(one) == 4 and one != untuned
    b.set_tuning(**reported)
    assert b.tuning() == reported and of_a_run(b, st) == untuned
    b.close()
    stream_destroy(st)


def test_autotuned_tuning_set_back_keeps_the_launches(hip):
    from hiprt import stream_create, stream_destroy
    print("[case] batch autotuned", flush=True)
    sizes = [(62, 55, 40), (31, 30, 29)]
    b, other, st = batch("f16s", sizes), batch("f16s", sizes), stream_create()
    b.autotune(trial_steps=2, stream=st)
    other.set_tuning(**b.tuning())
    got, want = of_a_run(b, st), of_a_run(other, st)
    assert got == want
    b.close()
    other.close()
    stream_destroy(st)
