"""Workloads that the performance of the framework is judged by: what a finite-element code has the engine do, through
the public entry points, on tensors that live on the GPU.

Every case is fp64 (the only type of the engine).  A case names a family and its sizes:

  reduction      the sum over a batch that the README opens with, ``S_i_j = A_n_i_j B_n``
  inverse        inverse and determinant of the Jacobians at every quadrature point
  assembly       element mass matrices, one kernel of seven operands
  mass           sum-factorised mass operator, seven kernels in one multi-kernel launch; "stored" keeps every
                 intermediate (a caller who only changes the policy string), otherwise they are marked transient
  diffusion      sum-factorised diffusion operator, eighteen kernels in one launch, slices, ``+=``
  mesh           the whole operator on a mesh of continuous elements: scatter, mass operator, sum-gather; "inside" says
                 whether the sum-gather is recorded in the launch with the rest or called after it
  geometry       geometric factors from the Jacobians, inverse and determinant recorded in the same launch
  interpolation  a dense table applied to every element vector (values at points) and its transpose (back)
"""
import functools
import math

import numpy as np
import torch

import acrotensor_amd as at
from acrotensor_amd import workloads

DEVICE = "cuda"


# ------------------------------------------------------------------------------------------------ the cases

def listed():
    return [
        # the smallest call: one kernel, a few hundred KB; nothing but latency, launches and host time
        {"name": "reduction_small", "family": "reduction", "n": 4096, "rows": 3, "cols": 3},
        # the README's kernel at the size of the baseline configuration
        {"name": "reduction_large", "family": "reduction", "n": 1 << 20, "rows": 3, "cols": 3},
        # Jacobians of 65536 elements with 64 quadrature points each
        {"name": "inverse_3x3", "family": "inverse", "elements": 65536, "points": 64, "dim": 3},
        # full assembly of quadratic hexahedra: written bytes dominate
        {"name": "assembly_p2", "family": "assembly", "elements": 32768, "p": 2, "q": 4},
        # one rank's share of a strong-scaled solve, an odd number of elements: a solver calls this thousands of times
        {"name": "mass_small", "family": "mass", "elements": 511, "p": 2, "q": 4, "stored": False},
        # the headline: cubic hexahedra, 2^24 degrees of freedom
        {"name": "mass_p3", "family": "mass", "elements": 262144, "p": 3, "q": 5, "stored": False},
        # the same operator of a caller who marks nothing as transient: every intermediate is a result
        {"name": "mass_p3_stored", "family": "mass", "elements": 65537, "p": 3, "q": 5, "stored": True},
        # the largest: degree 7, 33.5 million degrees of freedom, 5.3 GB of it geometric factors
        {"name": "diffusion_p7", "family": "diffusion", "elements": 65536, "p": 7, "q": 10},
        # an ordinary medium degree on a ragged number of elements
        {"name": "diffusion_p4", "family": "diffusion", "elements": 20011, "p": 4, "q": 6},
        # node vector to node vector on a ragged mesh
        {"name": "mesh_p3", "family": "mesh", "nx": 61, "ny": 64, "nz": 67, "p": 3, "q": 5, "inside": True},
        # set-up of the diffusion operator, once per mesh movement
        {"name": "geometry_q10", "family": "geometry", "elements": 16384, "q": 10},
        # cubic hexahedra: 64 coefficients to 125 points and back, on the matrix cores
        {"name": "interpolation_p3", "family": "interpolation", "elements": 131072, "points": 125, "coefficients": 64},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    family = rng.choice(["reduction", "inverse", "assembly", "mass", "mass", "diffusion", "mesh", "geometry", "interpolation"])
    if family == "reduction":
        return {"family": family, "n": _log_int(rng, 1 << 10, 1 << 22), "rows": rng.randint(2, 6), "cols": rng.randint(2, 6)}
    if family == "inverse":
        dim = rng.choice([2, 3, 3])
        return {"family": family, "elements": _log_int(rng, 1 << 8, 1 << 16), "points": rng.randint(2, 5) ** dim, "dim": dim}
    if family == "assembly":
        p = rng.randint(1, 3)
        q = p + rng.randint(1, 2)
        return {"family": family, "elements": _log_int(rng, 1 << 7, (1 << 25) // (p + 1) ** 6), "p": p, "q": q}
    if family == "mass":
        p = rng.randint(1, 8)
        stored = rng.random() < 0.25
        dofs = 1 << (22 if stored else 24)
        return {"family": family, "elements": _log_int(rng, 1 << 7, dofs // (p + 1) ** 3), "p": p, "q": p + rng.randint(1, 2), "stored": stored}
    if family == "diffusion":
        p = rng.randint(1, 8)
        q = p + rng.randint(1, 2)
        return {"family": family, "elements": _log_int(rng, 1 << 7, (1 << 25) // q ** 3), "p": p, "q": q}
    if family == "mesh":
        p = rng.randint(1, 4)
        edge = _log_int(rng, 6, 256 // (p + 1))
        nx, ny, nz = (max(2, int(edge * rng.uniform(0.7, 1.0))) for _ in range(3))
        return {"family": family, "nx": nx, "ny": ny, "nz": nz, "p": p, "q": p + rng.randint(1, 2), "inside": rng.random() < 0.5}
    if family == "geometry":
        q = rng.randint(2, 10)
        return {"family": family, "elements": _log_int(rng, 1 << 7, (1 << 24) // q ** 3), "q": q}
    p = rng.randint(1, 3)
    n = rng.choice([(p + 1) ** 3, rng.randint(8, 64)])
    return {"family": family, "elements": _log_int(rng, 1 << 8, 1 << 17), "points": rng.choice([(p + 2) ** 3, rng.randint(n, 128)]), "coefficients": n}


# ------------------------------------------------------------------------------------------------ building blocks

@functools.lru_cache(maxsize=None)
def _engine():
    """The engine of the program: it keeps what it has compiled, as a user's does."""
    return at.TensorEngine("HIP")


@functools.lru_cache(maxsize=1)
def _mesh(nx, ny, nz, p):
    """The mesh's element-to-node map: made once per mesh, whatever vectors are put through it."""
    dofs, nodes = workloads.hex_mesh_dof_map(nx, ny, nz, p)
    m = at.IndexMapping(nodes, dofs.size)
    m.map[:] = dofs.ravel()
    m.ComputeInverse()
    return m


def _wrap(t):
    """Engine tensor over a torch tensor's device memory (the host side is address space that nothing touches)."""
    return at.Tensor(*t.shape, hdata=np.empty(tuple(t.shape)), ddata=t.data_ptr(), ongpu=True)


class _State:
    def __init__(self, case, seed):
        self.case = case
        self.engine = _engine()
        self.generator = torch.Generator(DEVICE).manual_seed(int(seed))
        self.arrays, self.tensors, self.results = {}, {}, []

    def uniform(self, name, shape, lo, hi):
        a = torch.rand(shape, generator=self.generator, device=DEVICE, dtype=torch.float64)
        return self._add(name, a.mul_(hi - lo).add_(lo))

    def result(self, name, shape):
        self.results.append(name)
        return self._add(name, torch.empty(shape, device=DEVICE, dtype=torch.float64))

    def _add(self, name, a):
        self.arrays[name] = a
        self.tensors[name] = _wrap(a)
        return a

    def intermediate(self, name, shape, transient=True):
        t = at.Tensor(*shape)
        t.SetTransient(transient)
        t.SwitchToGPU()
        self.tensors[name] = t

    def slice(self, name, parent, i):
        self.tensors[name] = at.SliceTensor(self.tensors[parent], i)

    def outputs(self):
        return {name: self.arrays[name] for name in self.results}

    def launch(self, kernels):
        for k, names in kernels:
            self.engine(k, *[self.tensors[n] for n in names])


def _chain(*kernels):
    """(kernel string, variable names) of each kernel; the names of the tensors are the variables' own."""
    out = []
    for k in kernels:
        left, right = k.replace("+=", "=").split("=")
        out.append((k, [v.split("_")[0] for v in left.split() + right.split()]))
    return out


_MASS = _chain(
    "T1_e_q_j_k = B_q_i X_e_i_j_k",
    "T2_e_q_r_k = B_r_j T1_e_q_j_k",
    "T3_e_q_r_s = B_s_k T2_e_q_r_k",
    "U_e_q_r_s = D_e_q_r_s T3_e_q_r_s",
    "V1_e_i_r_s = B_q_i U_e_q_r_s",
    "V2_e_i_j_s = B_r_j V1_e_i_r_s",
    "Y_e_i_j_k = B_s_k V2_e_i_j_s")

_DIFFUSION = _chain(
    "T1g_e_q_j_k = G_q_i X_e_i_j_k",
    "T1b_e_q_j_k = B_q_i X_e_i_j_k",
    "T2a_e_q_r_k = B_r_j T1g_e_q_j_k",
    "T2b_e_q_r_k = G_r_j T1b_e_q_j_k",
    "T2c_e_q_r_k = B_r_j T1b_e_q_j_k",
    "U0_e_q_r_s = B_s_k T2a_e_q_r_k",
    "U1_e_q_r_s = B_s_k T2b_e_q_r_k",
    "U2_e_q_r_s = G_s_k T2c_e_q_r_k",
    "Z_m_e_q_r_s = D_e_q_r_s_m_n U_n_e_q_r_s",
    "V1a_e_i_r_s = G_q_i Z0_e_q_r_s",
    "V1b_e_i_r_s = B_q_i Z1_e_q_r_s",
    "V1c_e_i_r_s = B_q_i Z2_e_q_r_s",
    "V2a_e_i_j_s = B_r_j V1a_e_i_r_s",
    "V2b_e_i_j_s = G_r_j V1b_e_i_r_s",
    "V2c_e_i_j_s = B_r_j V1c_e_i_r_s",
    "Y_e_i_j_k = B_s_k V2a_e_i_j_s",
    "Y_e_i_j_k += B_s_k V2b_e_i_j_s",
    "Y_e_i_j_k += G_s_k V2c_e_i_j_s")

_REDUCTION = _chain("S_i_j = A_n_i_j B_n")
_ASSEMBLY = [("M_e_i_j_k_l_m_n = B_q_i B_q_l B_r_j B_r_m B_s_k B_s_n W_e_q_r_s", ["M"] + ["B"] * 6 + ["W"])]
_GEOMETRY = [("D_e_m_n_k1_k2_k3 = W_k1_k2_k3 C_e_k1_k2_k3 Jdet_e_k1_k2_k3 Jinv_e_k1_k2_k3_n_j Jinv_e_k1_k2_k3_m_j",
              ["D", "W", "C", "Jdet", "Jinv", "Jinv"])]
_INTERPOLATION = _chain("U_e_q = B_q_i X_e_i", "Y_e_i = B_q_i U_e_q")


def _mass_intermediates(E, P, Q):
    return {"T1": (E, Q, P, P), "T2": (E, Q, Q, P), "T3": (E, Q, Q, Q), "U": (E, Q, Q, Q), "V1": (E, P, Q, Q), "V2": (E, P, P, Q)}


def _elements(case):
    return case["nx"] * case["ny"] * case["nz"] if case["family"] == "mesh" else case["elements"]


# ------------------------------------------------------------------------------------------------ prepare and run

def prepare(case, seed):
    s = _State(case, seed)
    family = case["family"]
    if family == "reduction":
        n, r, c = case["n"], case["rows"], case["cols"]
        s.uniform("A", (n, r, c), 0.0, 1.0)
        s.uniform("B", (n,), 0.5, 1.5)
        s.result("S", (r, c))
    elif family == "inverse":
        E, q, d = case["elements"], case["points"], case["dim"]
        s.uniform("J", (E, q, d, d), -0.1, 0.1).diagonal(dim1=-2, dim2=-1).add_(1.0)
        s.result("Jinv", (E, q, d, d))
        s.result("Jdet", (E, q))
    elif family == "assembly":
        E, P, Q = case["elements"], case["p"] + 1, case["q"]
        s.uniform("B", (Q, P), -1.0, 1.0)
        s.uniform("W", (E, Q, Q, Q), 0.5, 1.5)
        s.result("M", (E, P, P, P, P, P, P))
    elif family in ("mass", "mesh"):
        E, P, Q = _elements(case), case["p"] + 1, case["q"]
        s.uniform("B", (Q, P), -1.0, 1.0)
        s.uniform("D", (E, Q, Q, Q), 0.5, 1.5)
        if family == "mesh":
            s.map = _mesh(case["nx"], case["ny"], case["nz"], case["p"])
            s.uniform("x", (s.map.domain_size,), -1.0, 1.0)
            s.intermediate("X", (E, P, P, P))
            s.intermediate("Y", (E, P, P, P), transient=False)
            s.result("y", (s.map.domain_size,))
        else:
            s.uniform("X", (E, P, P, P), -1.0, 1.0)
            s.result("Y", (E, P, P, P))
        for name, shape in _mass_intermediates(E, P, Q).items():
            (s.result if case.get("stored") else s.intermediate)(name, shape)
    elif family == "diffusion":
        E, P, Q = case["elements"], case["p"] + 1, case["q"]
        s.uniform("B", (Q, P), -1.0, 1.0)
        s.uniform("G", (Q, P), -1.0, 1.0)
        s.uniform("X", (E, P, P, P), -1.0, 1.0)
        D = s.uniform("D", (E, Q, Q, Q, 3, 3), -0.5, 0.5)        # symmetric and positive definite at every point
        for i in range(3):
            D[..., i, i].abs_().add_(1.1)
            for j in range(i):
                D[..., i, j].copy_(D[..., j, i])
        for name in ("T1g", "T1b"):
            s.intermediate(name, (E, Q, P, P))
        for x in "abc":
            s.intermediate("T2" + x, (E, Q, Q, P))
            s.intermediate("V1" + x, (E, P, Q, Q))
            s.intermediate("V2" + x, (E, P, P, Q))
        for name in "UZ":
            s.intermediate(name, (3, E, Q, Q, Q))
            for i in range(3):
                s.slice(name + str(i), name, i)
        s.result("Y", (E, P, P, P))
    elif family == "geometry":
        E, Q = case["elements"], case["q"]
        s.uniform("W", (Q, Q, Q), 0.1, 1.0)
        s.uniform("C", (E, Q, Q, Q), 0.5, 1.5)
        s.uniform("J", (E, Q, Q, Q, 3, 3), -0.1, 0.1).diagonal(dim1=-2, dim2=-1).add_(1.0)
        s.intermediate("Jinv", (E, Q, Q, Q, 3, 3))
        s.intermediate("Jdet", (E, Q, Q, Q))
        s.result("D", (E, 3, 3, Q, Q, Q))
    else:
        E, q, n = case["elements"], case["points"], case["coefficients"]
        s.uniform("B", (q, n), -1.0, 1.0)
        s.uniform("X", (E, n), -1.0, 1.0)
        s.result("U", (E, q))
        s.result("Y", (E, n))
    torch.cuda.synchronize()      # the inputs were made on torch's stream, the engine works on its own
    return s


def run(s):
    family, engine, t = s.case["family"], s.engine, s.tensors
    if family == "reduction":
        s.launch(_REDUCTION)
    elif family == "inverse":
        engine.BatchMatrixInvDet(t["Jinv"], t["Jdet"], t["J"])
    elif family == "assembly":
        s.launch(_ASSEMBLY)
    elif family == "mass":
        engine.BeginMultiKernelLaunch()
        s.launch(_MASS)
        engine.EndMultiKernelLaunch()
    elif family == "diffusion":
        engine.BeginMultiKernelLaunch()
        s.launch(_DIFFUSION)
        engine.EndMultiKernelLaunch()
    elif family == "mesh":
        engine.BeginMultiKernelLaunch()
        engine.FlatIndexedScatter(t["X"], t["x"], s.map)
        s.launch(_MASS)
        if s.case["inside"]:
            engine.FlatIndexedSumGather(t["y"], t["Y"], s.map)
        engine.EndMultiKernelLaunch()
        if not s.case["inside"]:
            engine.FlatIndexedSumGather(t["y"], t["Y"], s.map)
    elif family == "geometry":
        engine.BeginMultiKernelLaunch()
        engine.BatchMatrixInvDet(t["Jinv"], t["Jdet"], t["J"])
        s.launch(_GEOMETRY)
        engine.EndMultiKernelLaunch()
    else:
        s.launch(_INTERPOLATION)
    return s.outputs()


# ------------------------------------------------------------------------------------------------ work and tolerance

def work(case):
    """Bytes: every input once and every output once.  Flops: the sum-factorised count where there is one."""
    family = case["family"]
    if family == "reduction":
        n, m = case["n"], case["rows"] * case["cols"]
        return {"bytes": 8 * (n * m + n + m), "flops": 2 * n * m}
    if family == "inverse":
        n, d = case["elements"] * case["points"], case["dim"]
        return {"bytes": 8 * n * (2 * d * d + 1), "flops": n * (54 if d == 3 else 9)}
    if family == "assembly":
        E, P, Q = case["elements"], case["p"] + 1, case["q"]
        return {"bytes": 8 * (E * (Q ** 3 + P ** 6) + Q * P), "flops": 2 * E * (P ** 2 * Q ** 3 + P ** 4 * Q ** 2 + P ** 6 * Q)}
    if family in ("mass", "mesh"):
        E, P, Q = _elements(case), case["p"] + 1, case["q"]
        flops = E * (4 * Q * P * (P * P + Q * P + Q * Q) + Q ** 3)
        if family == "mesh":
            p = case["p"]
            nodes = (case["nx"] * p + 1) * (case["ny"] * p + 1) * (case["nz"] * p + 1)
            return {"bytes": E * (4 * P ** 3 + 8 * Q ** 3) + 16 * nodes + 8 * Q * P, "flops": flops + E * P ** 3}
        kept = sum(math.prod(shape) for shape in _mass_intermediates(E, P, Q).values()) if case["stored"] else 0
        return {"bytes": 8 * (E * (2 * P ** 3 + Q ** 3) + Q * P + kept), "flops": flops}
    if family == "diffusion":
        E, P, Q = case["elements"], case["p"] + 1, case["q"]
        return {"bytes": 8 * (E * (2 * P ** 3 + 9 * Q ** 3) + 2 * Q * P),
                "flops": E * (4 * (2 * Q * P ** 3 + 3 * Q * Q * P * P + 3 * Q ** 3 * P) + 18 * Q ** 3)}
    if family == "geometry":
        n = case["elements"] * case["q"] ** 3
        return {"bytes": 8 * (19 * n + case["q"] ** 3), "flops": n * (54 + 2 + 6 * 5 + 9)}
    E, q, n = case["elements"], case["points"], case["coefficients"]
    return {"bytes": 8 * (E * (2 * n + q) + q * n), "flops": 4 * E * q * n}


def tolerance(case):
    # Against the same path in extended precision every family shows a relative error of 0.7e-16 to 3.2e-16 and, over a
    # few thousand values, a largest one of up to 1.6e-15 (over the largest arrays, more): four times that, and some
    # room for the tail of the largest.
    return {"rel": 1.2e-15, "max": 2e-14}
