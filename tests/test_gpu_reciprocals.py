"""The device's arithmetic that starts from the hardware's reciprocal, over all
mantissas: the logarithm's quotient is the division's bit for bit (the CPU
build takes the division itself), and the reciprocal that chooses polygon
edges is within the 1 ULP that the CPU check of the choices allows it twice."""
import pytest

pytestmark = pytest.mark.gpu


def test_reciprocal_forms_over_all_mantissas(gpu_ctx):
    quotients, ulps = gpu_ctx.reciprocal_probe()
    print("quotients that differ: %d, reciprocal error %.4f x 2^-23" % (quotients, ulps), flush=True)
    assert quotients == 0
    # 1 ULP of a value in (1/2, 1], relative: at most 2^-23
    assert 0.0 < ulps <= 1.0
