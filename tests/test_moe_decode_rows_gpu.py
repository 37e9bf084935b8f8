"""The down launch of the one-token MoE layer where both decoders are codebook formats and the h rows that it stages, an
odd number of them of an odd number of 256s, end in half a group of the loads that write LDS directly: all parts of the
layer, the shared expert alone, the routed experts alone. Every launch follows the same launch of another layer: what a
launch leaves out would be found in LDS as that layer's values, not its own."""
import pytest

import oracle as O
from macseek_amd import quant as q
from test_moe_decode_gpu import SMALL_SHAPE_CHAIN_TOL, Layer
from util import up

pytestmark = pytest.mark.gpu

CASES = [  # (gate/up, down, shared, n_routed, dim, inter): all parts stage n_routed + 1 rows, Shared one, Routed n_routed
    (O.IQ1_S, O.IQ1_S, O.IQ2_XXS, 6, 2048, 1280),      # seven rows and one, a wave per row
    (O.IQ2_XXS, O.IQ2_XXS, O.IQ1_S, 6, 2048, 2304),    # the library's own inter: two waves per row, twelve in all
    (O.IQ1_S, O.IQ2_XXS, O.IQ2_XXS, 2, 512, 256),      # one group and a half
    (O.IQ2_XXS, O.IQ1_S, O.IQ1_S, 5, 2048, 768),       # Routed: five rows
    (O.IQ1_S, O.IQ1_S, O.IQ1_S, 0, 2048, 1280),        # a layer of the shared expert alone
]


@pytest.mark.parametrize("parts", [["All"], ["Gu", "Down"], ["Shared", "Routed"]], ids="+".join)
@pytest.mark.parametrize("gu,dn,sh,nr,dim,inter", CASES)
def test_odd_number_of_staged_rows(dev, gu, dn, sh, nr, dim, inter, parts):
    L, other = Layer(gu, dn, sh, nr, True, dim, inter), Layer(gu, dn, sh, nr, True, dim, inter, xscale=3.0, seed=500)
    y, y_other, e = up(L.y0.copy()), up(other.y0.copy()), q.Enc()
    t, t_other = L.table(), other.table()
    for p in parts:
        q.encode_moe_decode_table_part(e, other.args(y_other), q.Buffer.of(t_other), q.MoePart[p])
        q.encode_moe_decode_table_part(e, L.args(y), q.Buffer.of(t), q.MoePart[p])
    e.wait()
    # h enters the down launch as fp16: y is off by at most 2^-11 of the terms' sizes, and the less the fewer columns of h the
    # roundings average out over (smallest layer: 6.6e-5, whole chain 7.3e-5); a row's last values left out are off by 0.1 and more
    short = inter < 2048
    L.check(y, L.scratch, "+".join(parts), y_tol=2.0 ** -11 if short else 5e-5, chain_tol=SMALL_SHAPE_CHAIN_TOL if short else 5e-5)
