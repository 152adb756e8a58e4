"""Molecule / basis / shell-pair data model.

Mirrors the reference's data model (Util/structures.py) for the parts on the
integral + Fock-build path:

* ``ContractedGaussian``  Util/structures.py:834-856
* ``Atom``                Util/structures.py:807-828
* ``ShellPair`` / ``Shell`` Util/structures.py:918-968 (shell-pair quantities of
  Methods/c_ints/shellpair_quantities.c:5-38 computed with numpy here)
* ``Molecule``            Util/structures.py:319-523 (ground state only)
* ``read_input``          the INI input format, Util/structures.py:23-47

Besides the reference attributes, ``Molecule`` exposes flat shell tables
(``shell_table()``) that the HIP library consumes.
"""
import ast
import configparser
import json
import math
import os

import numpy as np

# Data/constants.py:2,6-9,31-36
TO_BOHR = 1.8897161646320724
N_ELECTRONS = {'H': 1, 'HE': 2, 'LI': 3, 'BE': 4, 'B': 5, 'C': 6, 'N': 7, 'O': 8, 'F': 9, 'NE': 10}
INTEGRAL_THRESHOLD = 1.0e-8
ENERGY_CONVERGENCE = 1.0e-7
LINEAR_DEPENDENCE = 1.0e-6
DIIS_MAX_CONDITION = 1.0e7

MAX_L = 2   # s, p, d shells


def ncart(l):
    return (l + 1) * (l + 2) // 2


def cart_components(l):
    """Cartesian components (lx, ly, lz), lx descending then ly descending
    (Methods/c_ints/angmom_index.c:3-15)."""
    return [(lx, ly, l - lx - ly) for lx in range(l, -1, -1) for ly in range(l - lx, -1, -1)]


# Data/transform_basis.py:3-12 (s, p identity; d rows on xx,xy,xz,yy,yz,zz).
# The reference runs under Python 2 without true division, so the last row's
# written `-1/2` is integer floor division and evaluates to -1: its fifth d
# function is zz - xx - yy (norm^2 7/3 for normalised components, with an
# r^2 s-type part), not the normalised 3zz - r^2 combination.  The same
# numbers are used here so that spherical-d results are the reference's.
_S3 = math.sqrt(3.0) / 2.0
CART_TO_SPHER = {
    0: np.array([[1.0]]),
    1: np.identity(3),
    2: np.array([[_S3, 0, 0, -_S3, 0, 0],
                 [0, 1, 0, 0, 0, 0],
                 [0, 0, 1, 0, 0, 0],
                 [0, 0, 0, 0, 1, 0],
                 [-1.0, 0, 0, -1.0, 0, 1]], dtype=float),
}

_BASIS_CACHE = None


def basis_library():
    global _BASIS_CACHE
    if _BASIS_CACHE is None:
        path = os.path.join(os.path.dirname(os.path.abspath(__file__)), "data", "basis_sets.json")
        with open(path) as fh:
            _BASIS_CACHE = json.load(fh)
    return _BASIS_CACHE


def remove_punctuation(basis_set):
    """Util/structures.py:975-977: '6-31G*' -> '631GS'."""
    return (basis_set.replace('*', 's').replace('-', '').replace('(', '').replace(')', '')
            .replace(',', '').upper())


class ContractedGaussian:
    """One contracted shell (Util/structures.py:834-856)."""

    def __init__(self, function, cartesian_l):
        self.AngularMomentum = int(function[0])
        if self.AngularMomentum > MAX_L:
            raise ValueError("shells above d are not supported (l=%d)" % self.AngularMomentum)
        self.NAngMomCart = ncart(self.AngularMomentum)
        self.NAngMomSpher = 2 * self.AngularMomentum + 1
        self.Primitives = [list(p) for p in function[1:]]
        self.NPrimitives = len(self.Primitives)
        self.Exponents = np.array([e for e, _ in self.Primitives], dtype=float)
        self.Coefficients = np.array([c for _, c in self.Primitives], dtype=float)
        self.DoubleExponents = 2.0 * self.Exponents
        l = self.AngularMomentum
        self.ScaledCCs = np.array([c * (2.0 * e) ** ((l + 1.5) / 2.0) for e, c in self.Primitives])
        if l in cartesian_l:
            self.NAngMom = self.NAngMomCart
            self.CartToSpher = np.identity(self.NAngMomCart)
            self.Spherical = False
        else:
            self.NAngMom = self.NAngMomSpher
            self.CartToSpher = CART_TO_SPHER[l]
            self.Spherical = l >= 2
        self.ContractionScaling = np.array(
            [(math.gamma(lx + 0.5) * math.gamma(ly + 0.5) * math.gamma(lz + 0.5)) ** -0.5
             for lx, ly, lz in cart_components(l)])


# Contracted shells depend only on (basis set, element, Cartesian l's), not
# on the atom's position: atoms of one element share the same (read-only)
# ContractedGaussian objects.
_SHELLS = {}


def _element_shells(basis_set, label, cartesian_l, lib):
    key = (basis_set, label, tuple(sorted(set(int(l) for l in cartesian_l))))
    shells = _SHELLS.get(key)
    if shells is None:
        shells = [ContractedGaussian(f, cartesian_l) for f in lib[basis_set][label]]
        _SHELLS[key] = shells
    return shells


class Atom:
    """Util/structures.py:807-828."""

    def __init__(self, index, row, basis_set, cartesian_l, to_bohr):
        label, Z, x, y, z = row
        self.Index = index
        self.Label = str(label).upper()
        self.NuclearCharge = float(Z)
        self.Coordinates = [x * to_bohr, y * to_bohr, z * to_bohr]
        lib = basis_library()
        if basis_set not in lib:
            raise KeyError("basis set %s not available" % basis_set)
        if self.Label not in lib[basis_set]:
            raise KeyError("element %s not in basis %s" % (self.Label, basis_set))
        self.Basis = list(_element_shells(basis_set, self.Label, cartesian_l, lib))
        self.NFunctions = sum(c.NAngMom for c in self.Basis)


class Shell:
    """Util/structures.py:963-968."""

    def __init__(self, coords, cgtf, index, index_vec):
        self.Coords = np.asarray(coords, dtype=float)   # shells of one atom share their centre's array
        self.Cgtf = cgtf
        self.Index = index
        self.Ivec = index_vec


class ShellPair:
    """Shell-pair quantities (Util/structures.py:918-956 with
    Methods/c_ints/shellpair_quantities.c:5-38)."""

    def __init__(self, coords_a, cgtf_a, ia, ia_vec, coords_b, cgtf_b, ib, ib_vec):
        self.Centre1 = Shell(coords_a, cgtf_a, ia, ia_vec)
        self.Centre2 = Shell(coords_b, cgtf_b, ib, ib_vec)
        A = np.array(coords_a, dtype=float)
        B = np.array(coords_b, dtype=float)
        a = cgtf_a.Exponents[:, None]
        b = cgtf_b.Exponents[None, :]
        sig = 1.0 / (a + b)
        r2 = float(np.dot(A - B, A - B))
        self.Ltot = cgtf_a.AngularMomentum + cgtf_b.AngularMomentum
        self.PrimitivePairSigmas = sig
        self.PrimitivePairOverlaps = (np.pi * sig) ** 1.5 * np.exp(-a * b * sig * r2)
        self.PrimitivePairCentres = (a[..., None] * A + b[..., None] * B) * sig[..., None]
        self.PrimitivePairHalfSigmas = 0.5 * sig
        self.CentreDisplacement = A - B
        self.Normalization = np.outer(cgtf_a.ContractionScaling, cgtf_b.ContractionScaling)
        self.ContractionCoeffs = np.outer(cgtf_a.ScaledCCs, cgtf_b.ScaledCCs)
        self.BasisTransform = np.kron(cgtf_a.CartToSpher, cgtf_b.CartToSpher)


# Molecule.shell_table's coordinate-free arrays per (basis, atom labels,
# Cartesian shells)
_SHELL_LAYOUTS = {}


class Molecule:
    """Ground-state molecule in a single basis (Util/structures.py:319-523).

    Two ways to build one:

    * the reference's ``Molecule(inputs, settings[, basis])``
      (Util/structures.py:321-332), ``inputs`` being the section reader of
      ``inputs_return_function``: Coords, Coords_Units, Charge, Multiplicity
      and Cartesian_L come from the input (Util/structures.py:335-384), the
      basis from ``basis`` or else ``settings.BasisSets[0]``;
    * ``Molecule(coords, basis=..., charge=..., multiplicity=...,
      cartesian_l=..., units=...)`` with ``coords`` rows ``[label, Z, x, y,
      z]``; units 'ANGSTROM' (default, scaled by TO_BOHR) or 'BOHR'/'ATOMIC'.

    ``States`` holds the ground state (Util/structures.py:551-556); excited
    states are not generated here.
    """

    def __init__(self, inputs=None, settings=None, basis=None, charge=0, multiplicity=1, cartesian_l=(),
                 units="ANGSTROM", build_pairs=False):
        if callable(inputs):
            coords, units, charge, multiplicity, cartesian_l = _molecule_inputs(inputs)
            self.ExcitationType = _excitation_type(inputs)
            if basis is None:
                if settings is None:
                    raise SystemExit("Error: Molecule(inputs, settings) needs the settings for its basis set")
                basis = settings.BasisSets[0]
        else:
            coords = inputs
            self.ExcitationType = None
            if coords is None:
                raise ValueError("Molecule needs coordinate rows or the reference's input reader")
            if basis is None:
                basis = "STO3G"
        self.Coords = [list(r) for r in coords]
        self.NAtom = len(coords)
        self.Charge = int(charge)
        self.Multiplicity = int(multiplicity)
        self.CartesianL = list(cartesian_l)
        self.CoordsScaleFactor = TO_BOHR if str(units).upper() == "ANGSTROM" else 1.0
        self.Basis = remove_punctuation(basis)
        self.Atoms = [Atom(i, r, self.Basis, self.CartesianL, self.CoordsScaleFactor)
                      for i, r in enumerate(self.Coords)]
        self.NElectrons = sum(N_ELECTRONS[a.Label] for a in self.Atoms) - self.Charge
        self.NOrbitals = sum(a.NFunctions for a in self.Atoms)
        self.NCgtf = sum(len(a.Basis) for a in self.Atoms)
        # Util/structures.py:484-492
        self.NAlphaElectrons = (self.NElectrons + (self.Multiplicity - 1)) // 2
        self.NBetaElectrons = (self.NElectrons - (self.Multiplicity - 1)) // 2
        if self.NAlphaElectrons - self.NBetaElectrons + 1 != self.Multiplicity or \
                self.NAlphaElectrons + self.NBetaElectrons != self.NElectrons:
            raise ValueError("charge and multiplicity inconsistent with specified molecule")
        # flat shell list in global order: atoms, then shells in basis order
        self.Shells = []
        off = 0
        for atom in self.Atoms:
            xyz = np.array(atom.Coordinates, dtype=float)
            for cg in atom.Basis:
                self.Shells.append(Shell(xyz, cg, len(self.Shells),
                                         list(range(off, off + cg.NAngMom))))
                off += cg.NAngMom
        self._shell_pairs = None
        if build_pairs:
            self.build_shell_pairs()
        self.Core = None
        self.Overlap = None
        self.NuclearRepulsion = None
        self._states = None
        self.NStates = 1

    @property
    def States(self):
        """Util/structures.py:551-560: the ground state, with its occupancy
        lists, made on first use (its n x n matrices cost more than the rest
        of the constructor, and a solve through ``hartree_fock.run`` does not
        read them)."""
        if self._states is None:
            n = self.NOrbitals
            self._states = [ElectronicState([1] * self.NAlphaElectrons + [0] * (n - self.NAlphaElectrons),
                                            [1] * self.NBetaElectrons + [0] * (n - self.NBetaElectrons), n)]
        return self._states

    @States.setter
    def States(self, states):
        self._states = states

    def build_shell_pairs(self):
        """All pairs a <= b (Util/structures.py:509-522)."""
        sp = {}
        for a, sa in enumerate(self.Shells):
            for b in range(a, len(self.Shells)):
                sb = self.Shells[b]
                sp[(a, b)] = ShellPair(sa.Coords, sa.Cgtf, a, sa.Ivec, sb.Coords, sb.Cgtf, b, sb.Ivec)
                sp[(a, b)].Molecule = self
        self._shell_pairs = sp
        return sp

    @property
    def ShellPairs(self):
        """Python ShellPair objects (built on first use; the HIP engine builds
        its own device-side pair data)."""
        if self._shell_pairs is None:
            self.build_shell_pairs()
        return self._shell_pairs

    # ------------------------------------------------------------------ #
    def shell_layout(self):
        """The arrays of ``shell_table`` that do not hold coordinates: they
        depend only on the basis, the atoms' labels in order and the Cartesian
        shells, and are built once per such layout (molecules of a batch share
        a handful of layouts).  Shared: not to be written to."""
        key = (self.Basis, tuple(a.Label for a in self.Atoms), tuple(self.CartesianL))
        lay = _SHELL_LAYOUTS.get(key)
        if lay is None:
            ns = len(self.Shells)
            l = np.array([s.Cgtf.AngularMomentum for s in self.Shells], dtype=np.int32)
            nprim = np.array([s.Cgtf.NPrimitives for s in self.Shells], dtype=np.int32)
            prim_off = np.zeros(ns, dtype=np.int32)
            prim_off[1:] = np.cumsum(nprim)[:-1]
            spher = np.array([1 if s.Cgtf.Spherical else 0 for s in self.Shells], dtype=np.int32)
            exps = np.concatenate([s.Cgtf.Exponents for s in self.Shells]).astype(float)
            cc = np.concatenate([s.Cgtf.ScaledCCs for s in self.Shells]).astype(float)
            ao_off = np.array([s.Ivec[0] for s in self.Shells], dtype=np.int32)
            nfun = np.array([len(s.Ivec) for s in self.Shells], dtype=np.int32)
            cart_off = np.zeros(ns, dtype=np.int32)
            nc = np.array([ncart(int(x)) for x in l], dtype=np.int32)
            cart_off[1:] = np.cumsum(nc)[:-1]
            per_atom = np.array([len(a.Basis) for a in self.Atoms], dtype=np.int64)
            lay = dict(nshell=ns, l=l, nprim=nprim, prim_off=prim_off, spher=spher, exps=exps, cc=cc,
                       ao_off=ao_off, nfun=nfun, cart_off=cart_off, ncart_total=int(nc.sum()), per_atom=per_atom)
            _SHELL_LAYOUTS[key] = lay
        return lay

    def shell_table(self):
        """Flat per-shell arrays consumed by the HIP library and the oracle
        (the caller's own copies)."""
        lay = self.shell_layout()
        xyz = np.array([a.Coordinates for a in self.Atoms], dtype=float)
        center = np.ascontiguousarray(np.repeat(xyz, lay["per_atom"], axis=0).reshape(-1))
        out = {k: (v.copy() if isinstance(v, np.ndarray) else v) for k, v in lay.items() if k != "per_atom"}
        out.update(center=center, nao=int(self.NOrbitals), natom=self.NAtom,
                   atom_xyz=np.ascontiguousarray(xyz.reshape(-1)),
                   atom_z=np.array([a.NuclearCharge for a in self.Atoms], dtype=float))
        return out

    def cart_to_final(self):
        """Matrix T (nao x ncart) with final-basis functions = T @ cartesian ones."""
        tab = self.shell_table()
        T = np.zeros((tab["nao"], tab["ncart_total"]))
        for s, sh in enumerate(self.Shells):
            o, c = tab["ao_off"][s], tab["cart_off"][s]
            m = sh.Cgtf.CartToSpher
            T[o:o + m.shape[0], c:c + m.shape[1]] = m
        return T


# ----------------------------------------------------------------------------
# Electronic states (Util/structures.py:862-916): numpy matrices as the
# reference's callers (MP2, properties, NOCI) read them.


class Matrices:
    """Util/structures.py:882-901: Occupancy, Density, Fock and, per spin,
    Exchange, MOs, Energies; the total holds the Coulomb matrix."""

    def __init__(self, n_orbitals, occupancy=(), total=False):
        self.Occupancy = list(occupancy)
        self.Density = np.zeros((n_orbitals, n_orbitals))
        self.Fock = np.zeros((n_orbitals, n_orbitals))
        if not total:
            self.Exchange = np.zeros((n_orbitals, n_orbitals))
            self.MOs = []
            self.Energies = []
        else:
            self.Coulomb = np.zeros((n_orbitals, n_orbitals))

    def sort_occupied(self):
        """Sort the occupied orbitals by energy (Util/structures.py:895-901)."""
        n = int(sum(self.Occupancy))
        idx = np.append(np.argsort(np.asarray(self.Energies)[:n]), np.arange(n, len(self.Occupancy)))
        self.Energies = np.asarray(self.Energies)[idx]
        self.MOs = np.asarray(self.MOs)[:, idx]


class ElectronicState:
    """Util/structures.py:862-876."""

    def __init__(self, alpha_occupancy, beta_occupancy, n_orbitals):
        total = [a + b for a, b in zip(alpha_occupancy, beta_occupancy)]
        self.NAlpha = int(sum(alpha_occupancy))
        self.NBeta = int(sum(beta_occupancy))
        self.S2 = None
        self.Energy = None
        self.TotalEnergy = None
        self.Total = Matrices(n_orbitals, occupancy=total, total=True)
        self.Alpha = Matrices(n_orbitals, occupancy=alpha_occupancy)
        self.Beta = Matrices(n_orbitals, occupancy=beta_occupancy)


# ----------------------------------------------------------------------------
# Input (Util/structures.py:23-305).  Errors end the run the way the
# reference's do: SystemExit with the reference's message (the reference
# prints it and calls sys.exit()).

_NO_DEFAULT = "__NO_DEFAULT__"
AVAILABLE_METHODS = [None, 'HF', 'MP2', 'MP2-SCS', 'NOCI', 'NOCI-P2', 'NOCI-P2-SCS', 'NOCI-P2-SOS', 'MP2-SOS']
AVAILABLE_REFERENCES = ['RHF', 'UHF', 'CUHF']
AVAILABLE_GUESSES = ['READ', 'CORE', 'SAD', 'MLP']


def inputs_return_function(section, parser):
    """Util/structures.py:32-47: ``inputs(name[, default])`` returns the
    section's value of ``name`` through ast.literal_eval, strings upper-cased;
    a missing key without a default raises configparser.NoOptionError."""
    def inputs(var_name, default=_NO_DEFAULT):
        var = default
        try:
            var = parser.get(section, var_name)
        except (configparser.Error, KeyError):
            pass
        if isinstance(var, str) and var == _NO_DEFAULT:
            raise configparser.NoOptionError(var_name, section)
        elif var is not default:
            var = ast.literal_eval(var)
        if isinstance(var, str):
            var = var.upper()
        return var
    return inputs


def _get(inputs, name, default):
    try:
        return inputs(name)
    except (configparser.Error, ValueError, SyntaxError):
        return default


class SetSCF:
    """Util/structures.py:189-247 (Set_SCF).  Guess also accepts "MLP" (the
    learned guess of this package); Loop = "HOST" (default: the reference's
    sequence, diagonalising every cycle) or "DEVICE" (the iteration on the
    GPU, densities by purification; keyword SCF_Loop, not in the
    reference)."""

    def __init__(self, inputs, n_basis_sets, method):
        self.Reference = _get(inputs, "Reference", "UHF")
        if self.Reference not in AVAILABLE_REFERENCES:
            raise SystemExit("Error: Only the following references are available: %s" % AVAILABLE_REFERENCES)
        self.ConstrainExcited = _get(inputs, "Constrain_Excited", self.Reference == "CUHF")
        self.Guess = _get(inputs, "SCF_Guess", "CORE")
        if self.Guess not in AVAILABLE_GUESSES:
            self.Guess = "CORE"
        if self.Guess == "READ" or method is None:
            try:
                state = inputs("MO_Read_State")
                states = [str(i) for i in state] if isinstance(state, (list, tuple)) else [str(state)]
                mo_basis = remove_punctuation(inputs("MO_Read_Basis"))
            except (configparser.Error, ValueError, SyntaxError, AttributeError):
                raise SystemExit("Error: Must give details of files to read alpha and beta MOs from, using "
                                 "keywords MO_Read_Basis and MO_Read_State")
            self.AlphaMOFile = [mo_basis + '_' + st + '.alpha_MOs' for st in states]
            self.BetaMOFile = [mo_basis + '_' + st + '.beta_MOs' for st in states]
        self.MaxIter = _get(inputs, "Max_SCF_Iterations", 25)
        self.BasisFit = _get(inputs, "Basis_Fit", n_basis_sets != 1)
        self.Loop = _get(inputs, "SCF_Loop", "HOST")
        if self.Loop not in ("HOST", "DEVICE"):
            raise SystemExit("Error: SCF_Loop must be HOST or DEVICE")


class SetDIIS:
    """Util/structures.py:253-279 (Set_DIIS).  An unknown DIIS_Type is taken
    as C1 (the reference keeps the unknown name and then fails at the first
    extrapolation)."""

    def __init__(self, inputs, reference):
        self.Use = _get(inputs, "Use_DIIS", True)
        self.Size = _get(inputs, "DIIS_Size", 15)
        self.Type = _get(inputs, "DIIS_Type", "C1")
        if self.Type not in ("C1", "C2"):
            self.Type = "C1"
        self.Start = _get(inputs, "DIIS_Start", 1)
        self.MaxCondition = _get(inputs, "DIIS_Max_Condition", DIIS_MAX_CONDITION)
        self.Threshold = 0.0


class SetMOM:
    """Util/structures.py:285-305 (Set_MOM)."""

    def __init__(self, inputs):
        use = _get(inputs, "Use_MOM", None)
        if isinstance(use, bool):
            self.Use = use
        else:
            self.Use = (_get(inputs, "Excitations", None) is not None
                        or _get(inputs, "Alpha_Excitations", None) is not None)
        self.Reference = _get(inputs, "MOM_Reference", "FIXED")
        if self.Reference not in ("MUTABLE", "FIXED"):
            self.Reference = "FIXED"


class Settings:
    """System-independent input data (Util/structures.py:78-183).  MP2_type
    is optional here (default "AFTER"): the reference requires it
    (Util/structures.py:86-87) although none of its shipped inputs sets it."""

    def __init__(self, inputs, section_name):
        self.MP2_type = _get(inputs, "MP2_type", "AFTER")
        if self.MP2_type not in ("AFTER", "BEFORE"):
            raise SystemExit("Error: MP2_type must be AFTER or BEFORE")
        self.Method = _get(inputs, "Method", "HF")
        if self.Method not in AVAILABLE_METHODS:
            self.Method = "HF"
        self.JobType = _get(inputs, "Job_Type", "ENERGY")
        if self.JobType not in ("ENERGY", "PROPERTY"):
            self.JobType = "ENERGY"
        self.PropertyType = None
        if self.JobType == "PROPERTY":
            # Util/structures.py:117-130: a missing or malformed grid leaves
            # the property type unset (the reference's inner exit is caught by
            # its outer handler)
            prop = _get(inputs, "Property_Type", None)
            grid = _get(inputs, "Property_Grid", None)
            if prop == "SCATTERING" and isinstance(grid, list):
                self.PropertyType = prop
                self.PropertyGrid = grid
        basis_sets = _get(inputs, "Basis_Sets", None)
        if not (isinstance(basis_sets, list) and basis_sets and isinstance(basis_sets[0], str)):
            raise SystemExit("Error: must include Basis_Sets keyword followed by at least one basis set in a list")
        self.BasisSets = [remove_punctuation(b) for b in basis_sets]
        lib = basis_library()
        for b in self.BasisSets:
            if b not in lib:
                raise SystemExit("Error: basis set %s not recognised" % b)
        self.PrintLevel = _get(inputs, "Print_Level", "BASIC")
        if self.PrintLevel not in ('MINIMAL', 'BASIC', 'VERBOSE', 'DEBUG'):
            self.PrintLevel = "BASIC"
        dump = _get(inputs, "Dump_MOs", False)
        self.DumpMOs = dump if isinstance(dump, bool) else False
        self.OutFileName = str(section_name) + '.out'
        self.OutFile = None
        self.SectionName = section_name
        self.SCF = SetSCF(inputs, len(self.BasisSets), self.Method)
        self.DIIS = SetDIIS(inputs, self.SCF.Reference)
        self.MOM = SetMOM(inputs)


def _molecule_inputs(inputs):
    """Util/structures.py:335-384: coordinates, units, charge, multiplicity,
    Cartesian_L."""
    try:
        coords = inputs("Coords")
    except (configparser.Error, ValueError, SyntaxError):
        raise SystemExit("Error: coordinates not found in input file")
    if not (isinstance(coords, list) and coords and isinstance(coords[0], list) and len(coords[0]) == 5):
        raise SystemExit("Error: Coordinates must be specified in list of lists format")
    units = _get(inputs, "Coords_Units", "ANGSTROM")
    if units not in ('ANGSTROM', 'BOHR', 'ATOMIC'):
        units = "ANGSTROM"
    try:
        charge = inputs("Charge")
    except (configparser.Error, ValueError, SyntaxError):
        raise SystemExit("Error: must specify molecule charge using Charge =")
    try:
        mult = inputs("Multiplicity")
    except (configparser.Error, ValueError, SyntaxError):
        raise SystemExit("Error: must specify molecule multiplicity using Multiplicity =")
    cart = _get(inputs, "Cartesian_L", [])
    return coords, units, charge, mult, list(cart or [])


def _excitation_type(inputs):
    exc = _get(inputs, "Excitations", None)
    if exc is None and (_get(inputs, "Alpha_Excitations", None) is not None
                        or _get(inputs, "Beta_Excitations", None) is not None):
        exc = "CUSTOM"
    return exc


def process_input(section, parser):
    """Util/structures.py:23-30: (molecule, settings) for one INI section."""
    inputs = inputs_return_function(section, parser)
    settings = Settings(inputs, section)
    molecule = Molecule(inputs=inputs, settings=settings)
    if settings.SCF.BasisFit and molecule.CartesianL != []:
        raise SystemExit("Error: basis fitting currently not available for Cartesian basis functions")
    return molecule, settings


def read_input(path):
    """Every section of a reference-format INI file as (section, molecule,
    settings), through process_input."""
    parser = configparser.ConfigParser()
    if not parser.read(path):
        raise SystemExit("Error: cannot read input file %s" % path)
    jobs = []
    for section in parser.sections():
        molecule, settings = process_input(section, parser)
        jobs.append((section, molecule, settings))
    return jobs
