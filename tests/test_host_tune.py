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


CACHE = """
import tempfile
path = os.path.join(tempfile.mkdtemp(), "tune.txt")
d, p = small()
m, nb = d["mtxd"], 4
x, h = device_array(16 * m * nb), device_array(16 * m * nb)
i = p.info()
old = "0 %d %d %d %d %d %d %d 9 1 2 256 0 1 1" % (i["n1"], i["n2"], i["n3"], 2 * i["kd1"] + 1, i["ncol"], i["nanl"], nb)
open(path, "w").write(old + "\\n")
os.environ["CPWGPU_TUNE_CACHE"] = path
for _ in range(2):
    q = hk.Plan.from_inputs(d)
    fake.fake_clear()
    hk._check(hk.lib().cpwgpu_plan_tune(q._h, nb, x, m, h, m, hk.PREC_FP64, None))
    print(sum(e.startswith("launch") for e in log()))
lines = open(path).read().split("\\n")[:-1]
assert lines[0] == old and len(lines) == 2 and lines[1].startswith(" ".join(old.split()[:8])), lines
"""


def test_cache_lines_of_another_numbering_are_passed_over():
    timed, cached = (int(v) for v in run(CACHE).split())
    assert timed > 100 and cached < 10
