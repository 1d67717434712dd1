"""The reference driver's timers from per-call-site statistics."""
import miniafqmc_amd as m


def test_one_kernel_propagators_count_their_products():
    """Six substeps are 48 products of the propagator, run as eight launches
    each or as one."""
    products = {"prop_pw": (6, 1.0), "prop_taylor": (36, 5.0), "prop_ps": (6, 1.0)}
    for stats in (products, {"prop_fused": (6, 7.0)}, {"prop_fused_cols": (6, 7.0)}):
        assert m.reference_timers(stats)["Propagation"] == (48, 7.0)
