"""Per-phase timing of an instance whose CFL bound admits no substep count (on the CPU, over
the stand-in of the HIP runtime, whose kernels leave every bound at zero): its time is that
of the stage."""
import hip_stub

CODE = """
import block_forms
g, st, ro = block_forms.model("ens_2", "fp64")
g.set_state(st)
g.set_runoff(ro)
g.kernel_times(True)
nt, _ = g.ensemble_advance(86400.0, nt_cap=3)
result([int(nt.max()), g.instance_times().tolist()])
"""


def test_times_without_substeps(tmp_path):
    nt, ms = hip_stub.run(tmp_path, CODE)
    assert nt < 1 and ms == [1.0] * 6              # an interval of the stand-in is one millisecond
