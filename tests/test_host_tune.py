"""What the tuner compares, on the CPU: a kernel that is fast for a few applies and slow
once they follow each other without a wait (the clock that a loop of applies settles to)
must not be preferred to the default, whose time holds."""

from tests.fake_runtime import run

BODY = """
d, p = small()
m, nb = d["mtxd"], 4
x, h = device_array(16 * m * nb), device_array(16 * m * nb)
fake.fake_cost(b"k_plane", 100.0, 100.0, 0)
fake.fake_cost(b"k_plane_fastId", 50.0, 200.0, 60)   # variant 0
default = p.get_variant(hk.PREC_FP64, hk.TUNE_PLANE)
assert default != 0
hk._check(hk.lib().cpwgpu_plan_tune(p._h, nb, x, m, h, m, hk.PREC_FP64, None))
print(default, p.get_variant(hk.PREC_FP64, hk.TUNE_PLANE))
"""


def test_final_choice_holds_in_a_loop():
    default, chosen = run(BODY).split()
    assert chosen == default


def test_faster_kernel_is_kept():
    default, chosen = run(BODY.replace("50.0, 200.0, 60", "50.0, 50.0, 60")).split()
    assert chosen == "0"
