"""Algorithmic (compulsory) HBM bytes per kernel launch.

Bytes = distinct array entries a launch must read + entries it writes.
Static geometry and topology are counted; intermediate arrays are counted
only where they cross a kernel boundary in this design (the per-sub-edge and
per-edge flux buffers, the node-layer records).  One function per kernel
family (the names the library's timing events use), in terms of the mesh
sizes, so that the benchmark and the documentation use the same model.
FP64 reals are 8 bytes, indices 4 bytes; `real` is the size of the state
reals (8 for the FP64 path).

Per-stage conditional traffic (EGF at RK stage 3, UARD at stage 3, the
OBC and river branches) is left out: it is small and not every launch has it.
"""

R8 = 8
I4 = 4


def sizes(model):
    h = model.hdr
    ts = int(bool(h.p.temperature_active)) + int(bool(h.p.salinity_active))   # tracers a launch advances
    return dict(M=h.m, N=h.n, NE=h.ne, NCV=h.ncv, KB=h.kb, KBM1=h.kbm1,
                RSN=h.nring_sn, RVE=h.nring_ve, TS=ts, N2E=2 + ts + int(not h.p.barotropic))


# ----------------------------------------------------------------- 2-D mode
def ext_momentum(s, real=R8):
    """One RK stage by element tile (k_ext_stage): elevation, edge terms and
    momentum in one launch.  Each element's, edge's and node's constants and
    state once; a tile's halo (about 0.35 records, 0.26 edges and 0.15 nodes
    per element again) is traffic, not counted here."""
    M, N, NE, NCV = s["M"], s["N"], s["NE"], s["NCV"]
    reads = (N * (4 * I4 + 10 * real)                  # neighbours; A1U, A2U, ART, CC_HVC
             + N * (4 * I4 + 12 * real + 6 * real)     # flags; EPOR .. DLTYE; ADX2D .. WVBOT
             + N * (2 + 3 + 1 + 2) * real              # UA, VA; UARK, VARK, ELRK1; D1; wind stress
             + NE * (I4 + 6 * real)                    # edge slots; edge geometry
             + M * (4 * I4 + 5 * real) + 2 * NCV * I4  # node flags; ART1, H, ELRK, EL, D; sub-edge lists
             + NCV * real)                             # EXTEL terms
    writes = N * 4 * real + NCV * real + M * 2 * real  # UA, VA, EL1, D1; next EXTEL terms; EL, D
    return reads + writes


# ----------------------------------------------------------------- 3-D mode
def _cvrecflux(s, layers, own, fields, uv_layers, bottom_records, real):
    """Records formed in LDS and face fluxes of `fields` fields in one launch:
    the ring and element geometry, VISCOFH and the velocities are read once,
    `own` node fields of each field (itself, its mean) read and its face
    fluxes (and the bottom layer's records for the tracer) written; no other
    node-layer record crosses HBM."""
    M, N, NCV, RSN = s["M"], s["N"], s["NCV"], s["RSN"]
    reads = (RSN * (1 + 2 * real) + M * (2 * I4 + 2 * real)    # ring slots and factors, NTSN, ART2, NN_HVC
             + M * layers * real                               # VISCOFH
             + fields * own * M * layers * real                # field, mean
             + 2 * N * I4 + M * 32 // 10 * I4                  # block element lists and local indices; the blocks' nodes (about 1.3 per node) and with their rings (1.9)
             + NCV * (3 * I4 + 6 * real) + N * real            # sub-edge geometry, DT1
             + N * uv_layers * 2 * real)                       # U, V
    writes = fields * (NCV * layers * real + (M * 8 * real if bottom_records else 0))
    return reads + writes


def cvrecflux_ts(s, real=R8):
    """ADV_T and ADV_S records and face fluxes in one launch."""
    return _cvrecflux(s, s["KBM1"], 2, s["TS"], s["KBM1"], True, real)


def cvrecflux_q(s, real=R8):
    """ADV_Q records and face fluxes of Q2 and Q2L in one launch."""
    return _cvrecflux(s, s["KBM1"] - 1, 1, 2, s["KBM1"], False, real)


def adv_ts(s, real=R8):
    """Ordered sub-edge sums + vertical flux + update of T and S."""
    M, NCV, KB, KBM1 = s["M"], s["NCV"], s["KB"], s["KBM1"]
    reads = (M * (3 * I4 + 4 * real) + 2 * NCV * I4 + M * (I4 + real)   # counts, flags; ART1, DT, DTFA, NN_HVC; slot lists; bottom VISCOFH
             + M * KB * real                                   # WTS
             + s["RSN"] * I4                                   # FCT rings
             + s["TS"] * (NCV * KBM1 * real                    # face fluxes
                          + M * KBM1 * real                    # F1
                          + M * 8 * real))                     # bottom record
    writes = s["TS"] * (M * KBM1 * real + 3 * M * real)        # FF; PFPXB, PFPYB, AH_BOTTOM
    return reads + writes


def adv_q(s, real=R8):
    """Ordered sub-edge sums + vertical flux + update of Q2 and Q2L."""
    M, NCV, KB, KBM1 = s["M"], s["NCV"], s["KB"], s["KBM1"]
    reads = (M * (I4 + 3 * real) + 2 * NCV * I4 + M * KB * real + s["RSN"] * I4
             + 2 * (NCV * (KBM1 - 1) * real + M * KB * real))
    writes = 2 * M * KB * real
    return reads + writes


def _uv_blk(s, real, uv):
    """ADVECTION / ADV_UV by element block: the element and edge data, the
    velocities of each layer once, and the outputs; records and edge terms
    stay in LDS."""
    M, N, NE, KB, KBM1 = s["M"], s["N"], s["NE"], s["KB"], s["KBM1"]
    reads = (NE * (5 * I4 + 4 * real)                  # IEC, IENODE, ISBC; XIJC, YIJC, DLTXC, DLTYC
             + N * (3 * I4 + 12 * real)                # NBE; A1U, A2U, XC, YC, ART, CC_HVC
             + N * (4 * I4 + 2 * real)                 # edge list, IUCP/ISBCE, river offset; EPOR, ...
             + N * 7 * I4                              # block tables: records, edges (about two per element each), edge slots
             + M * real                                # DT
             + N * KBM1 * 2 * real)                    # U, V
    if uv:
        reads += (N * 5 * real + M * real               # DT1, D1, COR, GRAV_E, ART; EGF
                  + N * KBM1 * 2 * real + N * KB * real)  # DRHOX, DRHOY; W
        writes = N * KBM1 * 3 * real + N * real        # UF, VF, VISCOFM
    else:
        writes = 2 * N * real                          # ADX2D, ADY2D
    return reads + writes


def adv3d_blk(s, real=R8):
    """ADVECTION_EDGE_GCN by element block, summed into ADX2D/ADY2D."""
    return _uv_blk(s, real, False)


def advuv_blk(s, real=R8):
    """ADV_UV_EDGE_GCN by element block -> UF, VF, VISCOFM."""
    return _uv_blk(s, real, True)


def vertvl(s, real=R8):
    """VERTVL_EDGE by node tile: the elements' sub-edge geometry and U, V,
    the nodes' sub-edge positions, column integral, correction."""
    M, N, NCV, KB, KBM1 = s["M"], s["N"], s["NCV"], s["KB"], s["KBM1"]
    reads = (2 * NCV * I4 + M * (3 * I4 + 6 * real)   # sub-edge positions; counts, flags, ART1, D, DT, ELF, H
             + N * (I4 + 7 * real)                    # tile element lists; DT1, DLTXE/DLTYE of 3 sub-edges
             + N * KBM1 * 2 * real)                   # U, V
    writes = M * KB * real + M * real                 # WTS, DTFA
    return reads + writes


def viscofh(s, real=R8):
    """VISCOF_H: nodal strain rate from the element ring."""
    M, N, KBM1, RVE = s["M"], s["N"], s["KBM1"], s["RVE"]
    reads = RVE * (I4 + 4 * real) + M * (3 * I4 + real) + N * KBM1 * 2 * real
    writes = M * KBM1 * real
    return reads + writes


def vdif_q(s, real=R8):
    """VDIF_Q (MY2.5): column solves for Q2, Q2L and the mixing coefficients,
    then Q2 = Q2F, Q2L = Q2LF.  Reads Q2 Q2L RHO1 KQ KM KH Q2F Q2LF and the
    ring of U/V; writes Q2F Q2LF Q2 Q2L L KM KH KQ.  The in-kernel scratch
    (elimination coefficients, VHP parked in Q2F/Q2LF) is not counted."""
    M, N, KB, KBM1, RVE = s["M"], s["N"], s["KB"], s["KBM1"], s["RVE"]
    reads = M * KB * 8 * real + N * KBM1 * 2 * real + RVE * I4 + M * 4 * real + N * 4 * real
    writes = M * KB * 8 * real
    return reads + writes


def vdif_uv(s, real=R8):
    """VDIF_UV: implicit vertical diffusion of UF and VF."""
    N, KB, KBM1 = s["N"], s["KB"], s["KBM1"]
    return N * KB * 3 * real + N * 6 * real + N * KBM1 * 2 * real + N * 3 * real


def vdif_ts(s, real=R8):
    """VDIF_TS: implicit vertical diffusion of T and S."""
    M, KB, KBM1 = s["M"], s["KB"], s["KBM1"]
    return M * KB * real + M * 5 * real + s["TS"] * (M * 2 * KBM1 * real + M * 3 * real)


def step_end(s, real=R8):
    """T1 = TF1, S1 = SF1 with DENS2 of them, U = UF, V = VF and the 2-D state."""
    M, N, KB = s["M"], s["N"], s["KB"]
    return M * KB * (2 * s["TS"] + (s["N2E"] > 2 + s["TS"])) * real + 4 * N * KB * real + (M + N) * 4 * real


def n2e3d(s, real=R8):
    """N2E3D of node-layer fields (KB layers): element means of their nodes;
    the mean of its two launches, of W and of KM1, T, S and RHO."""
    M, N, KB = s["M"], s["N"], s["KB"]
    return N * 3 * I4 + (s["N2E"] * (M * KB * real + N * KB * real)) // 2


FAMILIES = {f.__name__: f for f in (
    ext_momentum, cvrecflux_ts, cvrecflux_q,
    adv_ts, adv_q,
    adv3d_blk, advuv_blk, vertvl, viscofh, vdif_q, vdif_uv, vdif_ts,
    step_end, n2e3d)}


def bytes_per_launch(name, model, real=R8):
    return FAMILIES[name](sizes(model), real)
