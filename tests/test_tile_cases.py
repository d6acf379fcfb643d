"""The cases of tile_cases.py launch every kernel that they are there for: the
library's host code runs them on 256 compute units over a runtime that notes the
kernels' names (no GPU)."""
import stubbed


def test_cases_launch_every_kernel(tmp_path):
    stubbed.run(stubbed.build(tmp_path), r'''
import tile_cases as tc
stub.stub_kernels.restype = stub.stub_launched.restype = C.c_char_p
def wanted(*parts):
    return {k for k in stub.stub_kernels().decode().split() if any(p in k for p in parts)}
def launched():
    return set(stub.stub_launched().decode().split())
def dt(eq, n):
    return 0.1 / (n - 2) if eq == 2 else 1e-3

got = []
for eq, prec, n, steps in tc.PLANS:
    with sw.Plan(eq, n, dt(eq, n), precision=prec, algorithm=sw.TRAPEZOID, node_width=128) as p:
        launched()
        p.advance(steps)
        got.append(launched())
assert all(len(k) == 1 for k in got)
assert set().union(*got) == wanted("k_wide") and len(wanted("k_wide")) == 56

got = []
for eq, prec, n, steps in tc.BATCHES:
    one = np.full(1, eq, np.int32), np.full(1, n, np.int64), np.full(1, 1e-3), np.full(1, 0.5)
    with sw.Batch(*one, precision=prec) as b:
        launched()
        b.advance(steps)
        got.append(launched())
assert all(len(k) == 1 for k in got)
assert set().union(*got) == wanted("k_batch") and len(wanted("k_batch")) == 40

got = set()
for eq, bc, prec, W, n in tc.ROWS:
    with sw.Plan(eq, n, dt(eq, n), precision=prec, algorithm=sw.SWEPT, bc=bc, tpb=W, node_width=W) as p:
        p.set_profiling(True)
        launched()
        p.advance(tc.row_steps(eq, W))
        got |= launched()
assert wanted("k_heat_swept", "k_ks_swept", "k_euler_swept") <= got
assert not got & wanted("k_wide")

for eq, prec, alg, W, n in tc.PLAIN_ROWS:
    with sw.Plan(eq, n, dt(eq, n), precision=prec, algorithm=alg, tpb=W, node_width=W) as p:
        assert p.info()["node_width"] == W
        launched()
        p.advance(tc.row_steps(eq, W))
        assert len(launched() & wanted("k_heat_swept", "k_ks_swept", "k_euler_swept")) == 3, (eq, prec, alg, W, n)
print("done")
''')
