"""Face values that the edge EMFs read in the RK stages that share ring faces
(grmhd.hip emf_edge, face_line, with the neighbour table): restated here from
the kernel and compared with the face at the same position in the instance.
Every value must come from a full face (both transverse indices interior, which
its own block computes) or from a ring slot of the edge's block beyond an
outflow face, which the mask ring_own makes that block compute; the two speeds
from the faces on either side of the edge."""
import itertools

import pytest

from test_ring_push import neighbours

# extents, ghost layers, instances (blocks, first block, boundary: 1 periodic)
GRIDS = [
    ((8, 8, 8), 3, [((2, 3, 2), 0, (0,) * 6)]),
    ((5, 4, 3), 3, [((2, 2, 1), 0, (1, 1, 0, 0, 1, 1)), ((1, 2, 2), 4, (0,) * 6)]),
    ((4, 7, 4), 4, [((1, 1, 1), 0, (1,) * 6)]),
]


def face_line(m, n, ng, lo, hi, q):
    """(block, index) of the points m - 3 .. m + 2 along a direction of extent n; lo, hi: the neighbours or -1"""
    out = []
    for t in range(6):
        x = m + t - 3
        if t < 3 and x < ng and lo >= 0:
            out.append((lo, x + n))
        elif t >= 3 and x >= n + ng and hi >= 0:
            out.append((hi, x - n))
        else:
            out.append((q, x))
    return out


@pytest.mark.parametrize("n,ng,insts", GRIDS, ids=["outflow", "mixed", "self_periodic"])
def test_edges_read_their_own_faces(n, ng, insts):
    nq, nbr = neighbours(insts)
    blk = {}
    for nb, q0, bc in insts:
        for b in itertools.product(*(range(x) for x in nb)):
            blk[q0 + b[0] + nb[0] * (b[1] + nb[1] * b[2])] = (nb, q0, bc, b)

    def position(q, d, x):
        """index x of direction d in block q as a position in the instance (wrapped where periodic)"""
        nb, _, bc, b = blk[q]
        g = b[d] * n[d] + x - ng
        return g % (nb[d] * n[d]) if bc[2 * d] == 1 else g

    for q in range(nq):
        bc = blk[q][2]
        own = [nbr[(q, s)] < 0 and bc[s] != 1 for s in range(6)]     # the mask ring_own
        for C in range(3):
            P, Q = (C + 1) % 3, (C + 2) % 3
            # v^Q of the faces normal to P, along Q (and the other way round)
            for F, A in ((P, Q), (Q, P)):
                for m in range(ng, n[A] + ng + 1):
                    line = face_line(m, n[A], ng, nbr[(q, 2 * A)], nbr[(q, 2 * A + 1)], q)
                    for t, (qb, x) in enumerate(line):
                        want = m + t - 3
                        assert position(qb, A, x) == position(q, A, want)
                        # the other two directions of the face are the edge's own
                        assert all(blk[qb][3][d] == blk[q][3][d] for d in (C, F)) and blk[qb][1] == blk[q][1]
                        if ng <= x < n[A] + ng:
                            continue                                    # a full face of block qb
                        assert qb == q and own[2 * A + (x >= n[A] + ng)]  # its ring slot
                    # the speeds: points 2 and 3 of the same line
                    assert [position(b, A, x) for b, x in line[2:4]] == [position(q, A, m - 1), position(q, A, m)]
