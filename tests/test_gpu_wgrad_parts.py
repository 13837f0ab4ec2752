"""The weight gradient on both sides of its change from atomics to partial sums (64 additions
per element or 2^18 in all), against the CPU float64 oracle with test_gpu_wgrad.py's bound."""
import pytest

from test_gpu_wgrad import _case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,dims,cin_p,cout,taps", [
    (1, (16, 32, 32), 16, 16, 27),   # 64 parts, 458752 additions: atomics
    (1, (16, 32, 40), 16, 16, 27),   # 80 parts: partial sums
    (2, (12, 32, 40), 48, 16, 27),   # 120 parts, dY shifted
    (1, (5, 65, 66), 32, 24, 27),    # 162 parts, ragged
    (1, (16, 32, 32), 16, 1, 1),     # 256 parts of four wavefronts, few additions: atomics
    (1, (20, 40, 64), 32, 40, 1),    # 800 parts, one tap: partial sums
])
def test_both_ways(N, dims, cin_p, cout, taps):
    run, verify = _case(N, dims, cin_p, cout, taps, 7)
    print("wgrad", N, dims, cin_p, cout, taps, flush=True)
    run()
    verify(1)
    run()
    verify(2)
