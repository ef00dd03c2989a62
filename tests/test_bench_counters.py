"""bench.py finds the kernel of each pass among a profiler's names, whichever
of the pass's kernels the mesh and the precision have run."""
import pytest

import bench

LARGE = {"void k_elem<2, true, false>(snh::StepArgs)": 8, "void k_elem<2, false, false>(snh::StepArgs)": 4,
         "void k_elem_seq<2, true, false>(snh::StepArgs)": 4, "void k_node<false, false>(snh::StepArgs)": 8,
         "void k_node_tile<false, false>(snh::StepArgs)": 12, "k_geo(snh::StepArgs)": 5,
         "k_copy(double __vector(2) const*, double __vector(2)*, unsigned long)": 21}
SMALL = {"void k_elem<1, false, false>(snh::StepArgs)": 8, "void k_node_slot<false, 0>(snh::StepArgs)": 8,
         "void k_node_tile<false, false>(snh::StepArgs)": 12, "k_geo_tets(snh::StepArgs)": 5, "k_geo_batch(BatchGrid)": 9,
         "k_copy(double __vector(2) const*, double __vector(2)*, unsigned long)": 21}
MIXED = {"void k_elem_mx<4, true>(snh::StepArgs)": 16, "void k_elem_mx<4, false>(snh::StepArgs)": 4,
         "k_node_mx(snh::StepArgs)": 4, "k_geo(snh::StepArgs)": 5, "k_copy(double*)": 21}


@pytest.mark.parametrize("names,elem,node,geo", [(LARGE, "k_elem<2, true", "k_node<", "k_geo("),
                                                 (SMALL, "k_elem<1", "k_node_slot<", "k_geo_tets("),
                                                 (MIXED, "k_elem_mx<4, true", "k_node_mx(", "k_geo(")],
                         ids=["large", "small", "mixed"])
def test_kernel_of_each_pass(names, elem, node, geo):
    res = {n: [{"FETCH_SIZE": 1.0}] * k for n, k in names.items()}
    for prefix, want in (("k_elem", elem), ("k_node", node), ("k_geo", geo), ("k_copy", "k_copy(")):
        name, rows = bench._kernel_rows(res, prefix)
        assert want in name and len(rows) == names[name]
    assert bench._kernel_rows(res, "k_heat_elem") == (None, None)
