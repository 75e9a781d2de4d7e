"""Two blocks with a wall (block 1, eta = 0) and overset tables with receivers
of every kind that one launch of the boundary phase has to order."""
import numpy as np

DIMS = [(200, 160), (150, 70)]
WALL = (1, "wall_slip_kinematic", "+eta", "0", "-0", "0", "0", "0", "0")


def tables(nheld, nlate, nother, nuse=0, nface=0, twice=False, seed=0):
    """nheld receivers of block 1 that each other's stencils read; in block 0,
    nlate whose stencils reach the wall, nother that read none of them and nuse
    that read the held; nface on the wall itself, which it writes first and
    the late ones read.  twice: the first receiver is named again, with its
    donors, which leaves the values but takes the order away."""
    (ni, _), (n1, _) = DIMS
    recv, donor = [], []
    for q in range(nlate + nother + nuse):
        recv.append((0, (10 + q // 180) * ni + 10 + q % 180))
        row = 0 if q < nlate else 40 if q < nlate + nother else 9
        donor.append((1, row * n1 + 2 + q % 140))
    at = [(10 + q // 140, 5 + q % 140) for q in range(nheld)]
    for q in range(nheld):
        recv.append((1, at[q][0] * n1 + at[q][1]))
        a, b = at[(q + 7) % nheld]
        donor.append((1, (a - 2) * n1 + b - 2))
    for q in range(nface):
        recv.append((1, 3 * q + 1))
        donor.append((0, 100 * ni + 3 * q))
    coef = np.random.default_rng(seed).uniform(0.1, 1.0, (len(recv), 25))
    if twice:
        recv.append(recv[0])
        donor.append(donor[0])
        coef = np.concatenate([coef, coef[:1]])
    recv, donor = np.array(recv), np.array(donor)
    return dict(recv_block=recv[:, 0], recv_l=recv[:, 1], donor_block=donor[:, 0], donor_l=donor[:, 1],
                widths=np.array([[5, 5, 1]] * 2), coef=coef, hole_block=np.zeros(0, int), hole_l=np.zeros(0, int))
