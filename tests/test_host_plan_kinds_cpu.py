"""mq_host_plan_create refuses the kinds it does not know, with and without MQ_HOST_GATHER."""
import ctypes as C


def test_unknown_kinds_are_refused(oracle_engine):
    from qcmaquis_amd.desc import SiteDesc
    from qcmaquis_amd.gpu import lib
    from qcmaquis_amd.workload import centre_problem
    p = centre_problem(oracle_engine, 6, m=6)
    sd = SiteDesc(p.ham.symm, p.psi.phys, p.psi.left, p.psi.right, p.W, p.L.layout, p.R.layout)
    known = {0, 16}  # sigma, sigma with MQ_HOST_GATHER
    ok = set()
    for kind in list(range(4, 256)) + sorted(known):
        h = C.c_void_p()
        if lib().mq_host_plan_create(sd.ptr(), kind, C.byref(h)) == 0:
            ok.add(kind)
            lib().mq_host_plan_destroy(h)
    assert ok == known
