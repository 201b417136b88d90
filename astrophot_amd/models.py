"""Model classes with the reference's API (models/core_model.py,
model_object.py, galaxy_model_object.py, sersic_model.py, exponential_model.py,
gaussian_model.py, moffat_model.py, sky_model_object.py, flatsky_model.py,
group_model_object.py).

``AstroPhot_Model(model_type=...)`` dispatches on the ``model_type`` string
(core_model.py:98-115).  ``sample`` and ``jacobian`` run on the gfx950
kernels (see ``_engine``); the class attributes are the reference's knobs
(model_object.py:63-111) and keep its defaults.
"""

from __future__ import annotations

import io
import json
import math
from collections import OrderedDict
from typing import Optional, Sequence

import numpy as np
import torch
import yaml

from . import AP_config
from . import _engine
from . import _lib as L
from .errors import InvalidTarget, SpecificationConflict, UnrecognizedModel
from .image import Jacobian_Image, Model_Image, PSF_Image, Target_Image, Window
from .param import Param_Mask, Parameter_Node, _dval_drep1, _val_to_rep1

__all__ = ["AstroPhot_Model", "Component_Model", "Galaxy_Model", "Sersic_Galaxy", "Exponential_Galaxy",
           "Gaussian_Galaxy", "Moffat_Galaxy", "Sky_Model", "Flat_Sky", "PSF_Model", "Moffat_PSF",
           "Group_Model", "differentiable_sample"]


def _all_subclasses(cls):
    out = []
    for s in cls.__subclasses__():
        out.append(s)
        out.extend(_all_subclasses(s))
    return out


class AstroPhot_Model:
    """core_model.py:55-502."""

    model_type = "model"
    usable = False
    default_uncertainty = 1e-2

    def __new__(cls, *, model_type=None, filename=None, **kwargs):
        if filename is not None:  # core_model.py:98-106: the saved model_type picks the class
            model_type = AstroPhot_Model.load(filename)["model_type"]
        if model_type is not None:
            for M in _all_subclasses(AstroPhot_Model):
                if M.model_type == model_type and M.usable:
                    return super().__new__(M)
            raise UnrecognizedModel(f"Unknown AstroPhot model type: {model_type}")
        return super().__new__(cls)

    def __init__(self, *, name=None, target=None, window=None, locked=False, **kwargs):
        self.name = name if name is not None else f"{self.model_type}:{id(self)}"
        self.parameters = Parameter_Node(self.name)
        self._target = None
        self._target_identity = None
        self._window = None
        self.target = target
        self.window = window
        self.locked = locked
        self.mask = kwargs.get("mask", None)

    @classmethod
    def List_Models(cls, usable=None):
        out = _all_subclasses(AstroPhot_Model)
        return [m for m in out if usable is None or m.usable == usable]

    @property
    def target(self):
        return self._target

    @target.setter
    def target(self, tar):
        if not (tar is None or isinstance(tar, Target_Image)):
            raise InvalidTarget("AstroPhot_Model target must be a Target_Image instance.")
        self._target = tar
        if tar is not None:
            self._target_identity = tar.identity

    @property
    def window(self):
        """core_model.py:291-309."""
        if self._window is None:
            if self.target is None:
                raise ValueError("This model has no target or window, these must be provided by the user")
            return self.target.window.copy()
        return self._window

    @window.setter
    def window(self, window):
        """core_model.py:311-326."""
        if window is None:
            self._window = None
        elif isinstance(window, Window):
            self._window = window
        elif len(window) == 2:
            self._window = self.target.window.copy().crop_to_pixel(window)
        else:
            raise SpecificationConflict(f"Unrecognized window format: {window}")

    def make_model_image(self, window: Optional[Window] = None):
        """core_model.py:193-204."""
        w = self.window if window is None else (self.window & window)
        if type(self.target) is Target_Image:  # the window of target[w], without slicing its data
            return Model_Image(window=self.target.window & w)
        return self.target[w].model_image()

    def fit_mask(self):
        return torch.zeros_like(self.target[self.window].mask)

    def __call__(self, image=None, parameters=None, window=None, as_representation=False, **kwargs):
        """core_model.py:484-502."""
        if parameters is None:
            parameters = self.parameters
        elif isinstance(parameters, torch.Tensor):
            if as_representation:
                self.parameters.vector_set_representation(parameters)
            else:
                self.parameters.vector_set_values(parameters)
            parameters = self.parameters
        return self.sample(image=image, window=window, parameters=parameters, **kwargs)

    def __getitem__(self, key):
        return self.parameters[key]

    def __contains__(self, key):
        return key in self.parameters

    def initialize(self, target=None, parameters=None, **kwargs):
        pass

    # -- state on disk (core_model.py:374-449) ------------------------------
    def get_state(self, *args, **kwargs):
        return {"name": self.name, "model_type": self.model_type}

    def save(self, filename="AstroPhot.yaml"):
        """Write ``get_state()`` as YAML (.yaml) or JSON (.json)."""
        fname = str(filename)
        if fname.endswith(".yaml"):
            with open(fname, "w") as f:
                yaml.safe_dump(self.get_state(), f, indent=2)
        elif fname.endswith(".json"):
            with open(fname, "w") as f:
                json.dump(self.get_state(), f, indent=2)
        elif fname.endswith(".hdf5"):
            raise ValueError("hdf5 model files need h5py, which this installation lacks; use .yaml or .json")
        else:
            raise ValueError(f"Unrecognized filename format: {fname}, must be one of: .json, .yaml")

    @classmethod
    def load(cls, filename="AstroPhot.yaml"):
        """The state dictionary held by ``filename``: a dict, a text stream of
        YAML, or a .yaml / .json path.  YAML is read with the safe loader,
        which builds plain dicts, lists, strings and numbers only."""
        if isinstance(filename, dict):
            return filename
        if isinstance(filename, io.TextIOBase):
            return yaml.safe_load(filename)
        fname = str(filename)
        if fname.endswith(".yaml"):
            with open(fname, "r") as f:
                return yaml.safe_load(f)
        if fname.endswith(".json"):
            with open(fname, "r") as f:
                return json.load(f)
        raise ValueError(f"Unrecognized filename format: {fname}, must be one of: .json, .yaml "
                         "or a state dictionary")


class Component_Model(AstroPhot_Model):
    """model_object.py:25-444."""

    parameter_specs = {"center": {"units": "arcsec", "uncertainty": [0.1, 0.1]}}
    _parameter_order = ("center",)
    _profile = None
    psf_mode = "none"
    psf_convolve_mode = "fft"
    psf_subpixel_shift = "bilinear"
    sampling_mode = "midpoint"
    sampling_tolerance = 1e-2
    integrate_mode = "threshold"
    integrate_max_depth = 3
    integrate_gridding = 5
    integrate_quad_level = 3
    # integrate_mode "radius" (no reference counterpart): pixels whose centre
    # lies within this many pixels of the model centre take one
    # integrate_quad_level Gauss-Legendre level; the rest keep their sample
    integrate_radius = 5.0
    jacobian_chunksize = 10
    image_chunksize = 1000
    softening = 1e-3
    track_attrs = ["psf_mode", "psf_convolve_mode", "psf_subpixel_shift", "sampling_mode",
                   "sampling_tolerance", "integrate_mode", "integrate_max_depth", "integrate_gridding",
                   "integrate_quad_level", "integrate_radius", "jacobian_chunksize", "image_chunksize",
                   "softening"]

    def __init__(self, *, name=None, psf=None, parameters=None, **kwargs):
        super().__init__(name=name, **kwargs)
        self._psf = None
        if "filename" in kwargs:  # model_object.py:122-125
            self.load(kwargs["filename"], new_name=name)
            return
        for key in self.track_attrs:
            if key in kwargs:
                setattr(self, key, kwargs[key])
        if psf is not None:
            self.psf = psf
        specs = self.build_parameter_specs(parameters)
        for p in self._parameter_order:
            self.parameters.link(Parameter_Node(p, **specs[p]))
        if isinstance(parameters, torch.Tensor):
            self.parameters.vector_set_values(parameters)

    @classmethod
    def build_parameter_specs(cls, user_specs=None):
        """_model_methods.py:43-65."""
        specs = {}
        for base in reversed(cls.__mro__):
            if "parameter_specs" in base.__dict__:
                for k, v in base.__dict__["parameter_specs"].items():
                    specs[k] = dict(v)
        if isinstance(user_specs, dict):
            for p, v in user_specs.items():
                if isinstance(v, dict):
                    specs[p].update(v)
                else:
                    specs[p]["value"] = v
        return specs

    @property
    def psf(self):
        if self._psf is None:
            return None if self.target is None else self.target.psf
        return self._psf

    @psf.setter
    def psf(self, val):
        """model_object.py:158-174: a PSF_Image, a PSF model (re-rendered at
        every sample, its parameters joining this model's), or pixel data."""
        if val is None or isinstance(val, PSF_Image):
            self._psf = val
        elif isinstance(val, PSF_Model):
            self.set_aux_psf(val)
        else:
            self._psf = PSF_Image(data=val, pixelscale=self.target.pixelscale)

    def set_aux_psf(self, aux_psf, add_parameters=True):
        """model_object.py:133-147: ``aux_psf`` is sampled at every render of
        this model; with ``add_parameters`` its parameter node joins this
        model's tree (ahead of the model's own parameters when set at
        construction), so fits and Jacobians see the PSF parameters too."""
        self._psf = aux_psf
        if add_parameters:
            self.parameters.link(aux_psf.parameters)

    def _aux_psf(self):
        return self._psf if isinstance(self._psf, PSF_Model) else None

    # -- parameter bookkeeping for the engine ------------------------------
    def _values(self):
        return {k: n.value for k, n in self.parameters.nodes.items()}

    def _slot_of(self, name, element):
        if name == "center":
            return L.APX_P_CX + element
        if name in _engine.GEOM_SLOTS:
            return _engine.GEOM_SLOTS[name]
        return _engine.PROFILE_SLOTS[self._profile][name]

    def _free_slots(self):
        """(slot, dval/drep) for every element of the flat parameter vector.
        Parameters of an auxiliary PSF model take slot PSF_SLOT0 + their slot
        in the PSF model."""
        aux = self._aux_psf()
        aux_ids = set() if aux is None else {id(n) for n in aux.parameters._leaves()}
        out = []
        for leaf in self.parameters._leaves():
            values = leaf.value.reshape(-1).tolist()
            keep = None if leaf._mask is None else leaf._mask.reshape(-1).tolist()
            for e, v in enumerate(values):
                if keep is None or keep[e]:
                    rep = _val_to_rep1(v, *leaf.limits, leaf.cyclic)
                    d = _dval_drep1(rep, *leaf.limits, leaf.cyclic)
                    if id(leaf) in aux_ids:
                        out.append((_engine.PSF_SLOT0 + aux._slot_of(leaf.name, e), d))
                    else:
                        out.append((self._slot_of(leaf.name, e), d))
        return out

    # -- sampling (model_object.py:258-375) ---------------------------------
    def sample(self, image=None, window=None, parameters=None):
        if image is None:
            image = self.make_model_image(window=window)
        working_window = (image.window if window is None else window).copy()
        if "window" in self.psf_mode:
            raise NotImplementedError("PSF convolution in sub-window not available yet")
        if self.psf_convolve_mode not in ("fft", "direct"):
            raise ValueError(f"unrecognized psf_convolve_mode: {self.psf_convolve_mode}")
        if self.mask is None:
            _engine.render(self, self._values(), _engine.RenderRequest(window=working_window, image=image))
            return image
        # model_object.py:370-373: the mask zeroes this model's own samples
        # before they are added to the image
        part = Model_Image(window=working_window.copy())
        _engine.render(self, self._values(), _engine.RenderRequest(window=working_window, image=part))
        part.data *= self._keep(working_window)
        image += part
        return image

    def _keep(self, window):
        """1 where the model mask lets a sample of ``window`` through, else 0
        (float32, device); the mask covers the sampled window."""
        m = torch.as_tensor(self.mask, device=AP_config.ap_device)
        if tuple(m.shape) != (window.ny, window.nx):
            raise SpecificationConflict(
                f"{self.name}: mask shape {tuple(m.shape)} does not match the sampled window {(window.ny, window.nx)}")
        return torch.logical_not(m).to(torch.float32)

    def _mask_columns(self, jac, window, cols):
        """Zero this model's Jacobian columns ``cols`` at its masked pixels:
        the forward-mode derivative of the masked sample."""
        keep = self._keep(window)
        (dy, dx), (sy, sx), (h, w) = _engine._box(jac.window, window, window)
        for c in sorted(set(cols)):
            jac.data[dy:dy + h, dx:dx + w, c] *= keep[sy:sy + h, sx:sx + w]

    def _masked_G(self, G, G_window, window):
        """G with this model's masked pixels of ``window`` set to zero: the
        adjoint of the masked sample."""
        if self.mask is None:
            return G
        keep = self._keep(window)
        (dy, dx), (sy, sx), (h, w) = _engine._box(G_window, window, window)
        G = G.clone()
        G[dy:dy + h, dx:dx + w] *= keep[sy:sy + h, sx:sx + w]
        return G

    def jacobian(self, parameters: Optional[torch.Tensor] = None, as_representation: bool = False,
                 window: Optional[Window] = None, pass_jacobian: Optional[Jacobian_Image] = None, **kw):
        """_model_methods.py:260-396; writes straight into ``pass_jacobian``
        (the group's Jacobian) when given."""
        window = self.window if window is None else (self.window & window)
        if parameters is not None:
            if as_representation:
                self.parameters.vector_set_representation(parameters)
            else:
                self.parameters.vector_set_values(parameters)
        ids = self.parameters._identities()
        if pass_jacobian is None:
            jac = self.target[window].jacobian_image(parameters=list(self.parameters.vector_identities()))
        else:
            jac = pass_jacobian
            for pid in ids:
                if pid not in jac.parameters:
                    raise SpecificationConflict("pass_jacobian lacks this model's parameters")
        if len(ids) == 0:
            return jac
        slots = self._free_slots()
        slot_cols = {s: jac.parameters.index(pid) for (s, _), pid in zip(slots, ids)}
        dvdr = {s: (d if as_representation else 1.0) for s, d in slots}
        self._jacobian_windows(window, jac, slot_cols, dvdr)
        if self.mask is not None:
            self._mask_columns(jac, window, slot_cols.values())
        return jac

    def _jacobian_windows(self, window, jac, slot_cols, dvdr):
        """_chunk_image_jacobian (_model_methods.py:350-396) splits windows wider
        than image_chunksize; each piece renders on its own working grid."""
        nx, ny = window.nx, window.ny
        if max(nx, ny) > self.image_chunksize:
            ncx = int(math.ceil(nx / self.image_chunksize))
            ncy = int(math.ceil(ny / self.image_chunksize))
            csx, csy = int(round(nx / ncx)), int(round(ny / ncy))
            for ix in range(ncx):
                for iy in range(ncy):
                    sub = window.copy().crop_to_pixel(
                        [[csx * ix, min(nx, csx * (ix + 1))], [csy * iy, min(ny, csy * (iy + 1))]])
                    self._jacobian_windows(self.window & sub, jac, slot_cols, dvdr)
            return
        _engine.render(self, self._values(),
                       _engine.RenderRequest(window=window, jac=jac, slot_cols=slot_cols, dvdr=dvdr))

    def vjp(self, G, parameters: Optional[torch.Tensor] = None, as_representation: bool = True,
            window: Optional[Window] = None):
        """Vector-Jacobian product: sum over the model image of G * d image /
        d parameter, for this model's flat parameter vector (float64, device).
        ``G`` is a float32 image over ``window`` (default: this model's window).
        Runs the hand-written adjoint (``_engine.vjp``); nothing is stored from
        the forward pass."""
        if parameters is not None:
            if as_representation:
                self.parameters.vector_set_representation(parameters)
            else:
                self.parameters.vector_set_values(parameters)
        G_window = self.window if window is None else window
        G = torch.as_tensor(G, device=AP_config.ap_device).to(torch.float32).contiguous()
        n = len(self.parameters.vector_identities())
        if n == 0:
            return torch.zeros(0, dtype=torch.float64, device=AP_config.ap_device)
        slots = self._free_slots()
        slot_cols = {s: k for k, (s, _) in enumerate(slots)}
        dvdr = {s: (d if as_representation else 1.0) for s, d in slots}
        sample_window = self.window & G_window
        G = self._masked_G(G, G_window, sample_window)
        out, col_index = _engine.vjp(self, self._values(), sample_window, G, G_window, slot_cols, dvdr)
        return out[[col_index[k] for k in range(n)]]

    def get_state(self, save_params=True):
        """model_object.py:408-428: window, parameters (unless a group saves
        them), target identity, an image PSF, and the knobs that differ from
        the class defaults."""
        state = super().get_state()
        state["window"] = self.window.get_state()
        if save_params:
            state["parameters"] = self.parameters.get_state()
        state["target_identity"] = self._target_identity
        if isinstance(self._psf, (PSF_Image, PSF_Model)):
            state["psf"] = self._psf.get_state()
        for key in self.track_attrs:
            if getattr(self, key) != getattr(self.__class__, key):
                state[key] = getattr(self, key)
        return state

    def load(self, filename="AstroPhot.yaml", new_name=None):
        """_model_methods.py:437-482: name, window, knobs, parameters and an
        image PSF from a saved state.  The target is not saved; the one this
        model holds stays."""
        state = AstroPhot_Model.load(filename)
        self.name = state["name"] if new_name is None else new_name
        self.window = Window(**state["window"])
        self._target_identity = state.get("target_identity")
        self.target = self.target
        for key in self.track_attrs:
            if key in state:
                setattr(self, key, state[key])
        if isinstance(state["parameters"], Parameter_Node):
            self.parameters = state["parameters"]
        else:
            self.parameters = Parameter_Node(self.name, state=state["parameters"])
        missing = [p for p in self._parameter_order if p not in self.parameters.nodes]
        if missing:
            raise UnrecognizedModel(f"saved state of {self.name} lacks parameters {missing}")
        if "psf" in state:
            if state["psf"].get("type", "AstroPhot_Model") == "PSF_Image":
                self.psf = PSF_Image(state=state["psf"])
            else:  # _model_methods.py:473-482: the PSF model reads its branch of this tree
                sub = dict(state["psf"])
                sub["parameters"] = self.parameters[sub["name"]]
                self.set_aux_psf(AstroPhot_Model(name=sub["name"], filename=sub))
        return state


class Galaxy_Model(Component_Model):
    """galaxy_model_object.py:20-116."""

    model_type = f"galaxy {Component_Model.model_type}"
    parameter_specs = {
        "q": {"units": "b/a", "limits": (0, 1), "uncertainty": 0.03},
        "PA": {"units": "radians", "limits": (0, np.pi), "cyclic": True, "uncertainty": 0.06},
    }
    _parameter_order = Component_Model._parameter_order + ("q", "PA")


class Sersic_Galaxy(Galaxy_Model):
    """sersic_model.py:41-91."""

    model_type = f"sersic {Galaxy_Model.model_type}"
    parameter_specs = {
        "n": {"units": "none", "limits": (0.36, 8), "uncertainty": 0.05},
        "Re": {"units": "arcsec", "limits": (0, None)},
        "Ie": {"units": "log10(flux/arcsec^2)"},
    }
    _parameter_order = Galaxy_Model._parameter_order + ("n", "Re", "Ie")
    _profile = "sersic"
    usable = True

    def total_flux(self, parameters=None, window=None):
        p = self.parameters
        return _engine.sersic_total_flux(10 ** float(p["Ie"].value), float(p["n"].value),
                                         float(p["Re"].value), float(p["q"].value))


class Exponential_Galaxy(Galaxy_Model):
    """exponential_model.py:40-74."""

    model_type = f"exponential {Galaxy_Model.model_type}"
    parameter_specs = {"Ie": {"units": "log10(flux/arcsec^2)"}, "Re": {"units": "arcsec", "limits": (0, None)}}
    _parameter_order = Galaxy_Model._parameter_order + ("Re", "Ie")
    _profile = "exponential"
    usable = True


class Gaussian_Galaxy(Galaxy_Model):
    """gaussian_model.py:37-70."""

    model_type = f"gaussian {Galaxy_Model.model_type}"
    parameter_specs = {"sigma": {"units": "arcsec", "limits": (0, None)}, "flux": {"units": "log10(flux)"}}
    _parameter_order = Galaxy_Model._parameter_order + ("sigma", "flux")
    _profile = "gaussian"
    usable = True


class Moffat_Galaxy(Galaxy_Model):
    """moffat_model.py:23-68."""

    model_type = f"moffat {Galaxy_Model.model_type}"
    parameter_specs = {
        "n": {"units": "none", "limits": (0.1, 10), "uncertainty": 0.05},
        "Rd": {"units": "arcsec", "limits": (0, None)},
        "I0": {"units": "log10(flux/arcsec^2)"},
    }
    _parameter_order = Galaxy_Model._parameter_order + ("n", "Rd", "I0")
    _profile = "moffat"
    usable = True


class Sky_Model(Component_Model):
    """sky_model_object.py:6-35: centre locked, no PSF, no integration."""

    model_type = f"sky {Component_Model.model_type}"
    parameter_specs = {"center": {"units": "arcsec", "locked": True, "uncertainty": 0.0}}

    @property
    def psf_mode(self):
        return "none"

    def get_state(self, save_params=True):
        """group_model_object.py:325-337: the group's parameter tree, and each
        sub-model's state without its parameters (they sit in the tree)."""
        state = super().get_state()
        if save_params:
            state["parameters"] = self.parameters.get_state()
        state["models"] = {m.name: m.get_state(save_params=False) for m in self.models.values()}
        return state

    def load(self, filename="AstroPhot.yaml", new_name=None):
        """group_model_object.py:339-365: rebuild the parameter tree, then load
        each sub-model onto its branch (sub-models this group lacks are made
        from their saved model_type)."""
        state = AstroPhot_Model.load(filename)
        self.name = state["name"] if new_name is None else new_name
        if isinstance(state["parameters"], Parameter_Node):
            self.parameters = state["parameters"]
        else:
            self.parameters = Parameter_Node(self.name, state=state["parameters"])
        for mname, sub in state["models"].items():
            sub = dict(sub)
            sub["parameters"] = self.parameters[mname]
            if mname in self.models:
                self.models[mname].load(sub)
            else:
                self.add_model(AstroPhot_Model(name=mname, filename=sub, target=self.target))
        self.update_window()
        return state

    @psf_mode.setter
    def psf_mode(self, val):
        pass

    @property
    def integrate_mode(self):
        return "none"

    @integrate_mode.setter
    def integrate_mode(self, val):
        pass

    def __init__(self, **kwargs):
        super().__init__(**kwargs)
        if self.parameters["center"].value is None:
            self.parameters["center"]._value = self.window.center.clone()
            self.parameters["center"].shape = (2,)


class Flat_Sky(Sky_Model):
    """flatsky_model.py:12-55."""

    model_type = f"flat {Sky_Model.model_type}"
    parameter_specs = {"F": {"units": "log10(flux/arcsec^2)"}}
    _parameter_order = Sky_Model._parameter_order + ("F",)
    _profile = "flat_sky"
    usable = True


class PSF_Model(Component_Model):
    """psf_model_object.py:20-264: a model of the PSF itself.  Its target is a
    PSF_Image and its centre is fixed at the plane origin (the PSF image's
    centre pixel); it is sampled with Simpson's rule plus threshold
    integration by default, never convolved, and normalised to unit sum over
    the sampled window (``normalize_psf``)."""

    parameter_specs = {"center": {"units": "arcsec", "value": (0.0, 0.0), "uncertainty": (0.1, 0.1),
                                  "locked": True}}
    _parameter_order = ("center",)
    model_type = f"psf {AstroPhot_Model.model_type}"
    usable = False
    _is_psf = True
    normalize_psf = True
    sampling_mode = "simpsons"
    sampling_tolerance = 1e-3
    integrate_mode = "threshold"
    track_attrs = ["sampling_mode", "sampling_tolerance", "integrate_mode", "integrate_max_depth",
                   "integrate_gridding", "integrate_quad_level", "jacobian_chunksize", "softening"]

    def __init__(self, *, name=None, **kwargs):
        if "normalize_psf" in kwargs:
            self.normalize_psf = bool(kwargs["normalize_psf"])
        super().__init__(name=name, **kwargs)
        if "filename" not in kwargs and self._window is None and self.target is None:
            raise InvalidTarget("a PSF model needs a PSF_Image target or a window")
        c = self.window.center
        if float(c.abs().max()) > 1e-9 * float(self.window.pixel_length.max()):
            raise SpecificationConflict("PSF models must always be centered at (0,0)")

    @property
    def target(self):
        return self._target

    @target.setter
    def target(self, tar):
        if not (tar is None or isinstance(tar, PSF_Image)):
            raise InvalidTarget("PSF_Model target must be a PSF_Image instance.")
        self._target = tar
        if tar is not None:
            self._target_identity = tar.identity

    @property
    def psf_mode(self):
        return "none"

    @psf_mode.setter
    def psf_mode(self, val):
        if val != "none":
            raise SpecificationConflict("a PSF model is never convolved")

    @property
    def psf(self):
        return None

    @psf.setter
    def psf(self, val):
        if val is not None:
            raise SpecificationConflict("a PSF model is never convolved")

    def make_model_image(self, window: Optional[Window] = None):
        """psf_model_object.py:167-178."""
        w = self.window if window is None else (self.window & window)
        return Model_Image(window=w.copy())

    def fit_mask(self):
        return torch.zeros((self.window.ny, self.window.nx), dtype=torch.bool, device=AP_config.ap_device)

    def vjp(self, G, parameters: Optional[torch.Tensor] = None, as_representation: bool = True,
            window: Optional[Window] = None):
        """sum over the PSF image of G * d image / d parameter.  A PSF image is
        small (at most 129 x 129 pixels), so this contracts its Jacobian, the
        unit-sum normalisation included."""
        if window is not None and not window == self.window:
            raise SpecificationConflict("a PSF model's vjp covers its whole window")
        jac = self.jacobian(parameters=parameters, as_representation=as_representation).data
        G = torch.as_tensor(G, device=jac.device).to(torch.float64)
        return torch.einsum("yxk,yx->k", jac.double(), G)

    @property
    def psf_border_int(self):
        """The convolution border of the PSF this model renders (psf_image.py:71-93)."""
        return (int(math.ceil((1 + self.window.nx) / 2)), int(math.ceil((1 + self.window.ny) / 2)))


class Moffat_PSF(PSF_Model):
    """moffat_model.py:71-119: I(R) = 10**I0 / (1 + (R/Rd)^2)^n on the PSF
    plane, R = sqrt(x^2 + y^2 + softening^2)."""

    model_type = f"moffat {PSF_Model.model_type}"
    parameter_specs = {
        "n": {"units": "none", "limits": (0.1, 10), "uncertainty": 0.05},
        "Rd": {"units": "arcsec", "limits": (0, None)},
        "I0": {"units": "log10(flux/arcsec^2)", "value": 0.0, "locked": True},
    }
    _parameter_order = PSF_Model._parameter_order + ("n", "Rd", "I0")
    _profile = "moffat"
    usable = True


class Group_Model(AstroPhot_Model):
    """group_model_object.py:23-365."""

    model_type = f"group {AstroPhot_Model.model_type}"
    usable = True

    def __init__(self, *, name=None, models: Optional[Sequence[AstroPhot_Model]] = None, **kwargs):
        self.models = OrderedDict()
        super().__init__(name=name, **kwargs)
        if models is not None:
            self.add_model(models)
        self.update_window()
        if "filename" in kwargs:  # group_model_object.py:64-65
            self.load(kwargs["filename"], new_name=name)

    def add_model(self, model):
        if isinstance(model, (tuple, list)):
            for m in model:
                self.add_model(m)
            return
        if model.name in self.models and model is not self.models[model.name]:
            raise KeyError(f"{self.name} already has model with name {model.name}")
        self.models[model.name] = model
        self.parameters.link(model.parameters)
        if self.target is None:
            self._target = model.target
        self.update_window()

    def update_window(self, include_locked: bool = False):
        """group_model_object.py:92-129 (single target)."""
        w = None
        for m in self.models.values():
            if m.locked and not include_locked:
                continue
            w = m.window.copy() if w is None else (w | m.window)
        self._window = w

    @property
    def psf_mode(self):
        return "none"

    def get_state(self, save_params=True):
        """group_model_object.py:325-337: the group's parameter tree, and each
        sub-model's state without its parameters (they sit in the tree)."""
        state = super().get_state()
        if save_params:
            state["parameters"] = self.parameters.get_state()
        state["models"] = {m.name: m.get_state(save_params=False) for m in self.models.values()}
        return state

    def load(self, filename="AstroPhot.yaml", new_name=None):
        """group_model_object.py:339-365: rebuild the parameter tree, then load
        each sub-model onto its branch (sub-models this group lacks are made
        from their saved model_type)."""
        state = AstroPhot_Model.load(filename)
        self.name = state["name"] if new_name is None else new_name
        if isinstance(state["parameters"], Parameter_Node):
            self.parameters = state["parameters"]
        else:
            self.parameters = Parameter_Node(self.name, state=state["parameters"])
        for mname, sub in state["models"].items():
            sub = dict(sub)
            sub["parameters"] = self.parameters[mname]
            if mname in self.models:
                self.models[mname].load(sub)
            else:
                self.add_model(AstroPhot_Model(name=mname, filename=sub, target=self.target))
        self.update_window()
        return state

    def sample(self, image=None, window=None, parameters=None):
        """group_model_object.py:183-231.

        When the group allocates its own image, each component renders
        straight into it, clipped to the component's window: the reference's
        intermediate component image (model window & group window, zero plus
        the component) adds the same float values in the same order."""
        if image is None:
            sample_window = True
            image = self.make_model_image(window=window)
        else:
            sample_window = False
        if window is None:
            window = image.window
        if sample_window and image.window == window:
            for model in self.models.values():
                if isinstance(model, Component_Model) and model.mask is None:
                    _engine.render(model, model._values(),
                                   _engine.RenderRequest(window=window, image=image, region=model.window & window))
                else:
                    image += model(window=window)
            return image
        working = image[window].blank_copy()
        for model in self.models.values():
            if sample_window:
                working += model(window=window)
            else:
                model(working, window=window)
        image += working
        return image

    def jacobian(self, parameters: Optional[torch.Tensor] = None, as_representation: bool = False,
                 pass_jacobian: Optional[Jacobian_Image] = None, window: Optional[Window] = None, **kw):
        """group_model_object.py:233-283."""
        if window is None:
            window = self.window
        if parameters is not None:
            if as_representation:
                self.parameters.vector_set_representation(parameters)
            else:
                self.parameters.vector_set_values(parameters)
        jac = pass_jacobian
        if jac is None:
            jac = self.target[window].jacobian_image(parameters=list(self.parameters.vector_identities()))
        for model in self.models.values():
            model.jacobian(as_representation=as_representation, pass_jacobian=jac, window=window)
        return jac

    def vjp(self, G, parameters: Optional[torch.Tensor] = None, as_representation: bool = True,
            window: Optional[Window] = None):
        """Vector-Jacobian product of the group image (see Component_Model.vjp);
        components are sampled on the group window as in ``sample``."""
        if parameters is not None:
            if as_representation:
                self.parameters.vector_set_representation(parameters)
            else:
                self.parameters.vector_set_values(parameters)
        G_window = self.window if window is None else window
        G = torch.as_tensor(G, device=AP_config.ap_device).to(torch.float32).contiguous()
        parts = []
        for model in self.models.values():
            n = len(model.parameters.vector_identities())
            if n == 0:
                continue
            slots = model._free_slots()
            slot_cols = {sl: k for k, (sl, _) in enumerate(slots)}
            dvdr = {sl: (d if as_representation else 1.0) for sl, d in slots}
            Gm = model._masked_G(G, G_window, G_window) if isinstance(model, Component_Model) else G
            out, col_index = _engine.vjp(model, model._values(), G_window, Gm, G_window, slot_cols, dvdr,
                                         region=model.window & G_window)
            parts.append(out[[col_index[k] for k in range(n)]])
        return torch.cat(parts) if parts else torch.zeros(0, dtype=torch.float64, device=AP_config.ap_device)

    def fit_mask(self):
        return torch.zeros_like(self.target[self.window].mask)

    def __iter__(self):
        return iter(self.models.values())


class _RenderFunction(torch.autograd.Function):
    """model image as a differentiable function of the representation vector;
    backward is the hand-written adjoint (``model.vjp``)."""

    @staticmethod
    def forward(ctx, rep, model):
        ctx.model = model
        ctx.save_for_backward(rep)
        img = model(parameters=rep.detach().to("cpu", torch.float64), as_representation=True)
        return img.data.clone()

    @staticmethod
    def backward(ctx, G):
        (rep,) = ctx.saved_tensors
        g = ctx.model.vjp(G, parameters=rep.detach().to("cpu", torch.float64), as_representation=True)
        return g.to(device=rep.device, dtype=rep.dtype), None


def differentiable_sample(model, rep: torch.Tensor) -> torch.Tensor:
    """``model(parameters=rep, as_representation=True).data`` with autograd
    support through the gfx950 adjoint kernels."""
    return _RenderFunction.apply(rep, model)
