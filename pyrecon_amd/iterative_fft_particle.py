"""Drop-in ``OriginalIterativeFFTParticleReconstruction`` / ``IterativeFFTParticleReconstruction`` on MI355X
(pyrecon/iterative_fft_particle.py:9-245; Bautista et al. 2018).

Each iteration repaints the data at their current real-space estimate (wrapped), smooths, forms the
density contrast, transforms, divides by k^2 and reads the displacement at the data; the RSD part
of the displacement (reduced by beta / (1 + beta) in the first iteration) is then removed from the
original positions.  All of it runs in the HIP library, the per-point algebra with numpy's expressions
in the positions dtype; where numpy would promote beyond that dtype (f4 positions with a f8 mesh and a
global line of sight or wrap, or with a growth rate or bias that is a numpy f8), or for other dtypes, the
algebra is the reference's numpy on the host.
"""
import numpy as np

from . import _lib
from ._lib import lib, check
from .device import DeviceArray, as_device, device_view, stream_handle
from .mesh import RealMesh
from .recon import BaseReconstruction, SpectralReconstruction, ReconstructionError, _suffix, distance, keeps_class, \
    keeps_dtype, numpy_mean


class OriginalIterativeFFTParticleReconstruction(SpectralReconstruction):
    """Bautista et al. 2018 (pyrecon/iterative_fft_particle.py:9-239)."""

    def assign_data(self, positions, weights=None):
        """Paint the data and keep their positions (for :meth:`run`) and weights (iterative_fft_particle.py:16-31)."""
        view = device_view(positions)
        positions = view.numpy(stream=self.stream) if view is not None else np.asarray(positions)
        view = device_view(weights)
        if view is not None: weights = view.numpy(stream=self.stream)
        if weights is None:
            weights = np.ones_like(positions, shape=(len(positions),))
        if self.wrap: positions = self.info.wrap(positions)
        if self.mesh_data.buffer is None:
            self._positions_data = positions
            self._weights_data = weights
        else:
            self._positions_data = np.concatenate([self._positions_data, positions], axis=0)
            self._weights_data = np.concatenate([self._weights_data, weights], axis=0)
        self.mesh_data.assign_cic(positions, weights=weights, wrap=self.wrap)

    def set_density_contrast(self, ran_min=0.01, smoothing_radius=15.):
        """Density contrast of the (already smoothed) meshes (iterative_fft_particle.py:33-59); the data and
        randoms meshes are kept.  Sums are deterministic FP64."""
        self.ran_min = ran_min
        self.smoothing_radius = smoothing_radius
        dtype = self.info.dtype
        rtype = dtype.type
        delta = RealMesh(info=self.info, workspace=self.workspace, stream=self.stream)
        delta._allocate(zero=False)
        fn = getattr(lib, 'prh_density_contrast_' + _suffix(dtype))
        data = self.mesh_data.buffer
        if self.has_randoms:
            randoms = self.mesh_randoms.buffer
            s_data, s_randoms = self._mesh_sums(data, randoms)
            sum_data, sum_randoms = rtype(s_data), rtype(s_randoms)
            alpha = sum_data * 1. / sum_randoms
            threshold = ran_min * sum_randoms / self._size_randoms
            status = fn(data.ptr, randoms.ptr, delta.buffer.ptr, self.info.size, float(alpha), float(threshold),
                        float(self.bias * alpha), float(rtype(self.bias)), stream_handle(self.stream))
        else:
            s_data, _ = self._mesh_sums(data)
            mean = numpy_mean(rtype, s_data, self.info.size)
            status = fn(data.ptr, None, delta.buffer.ptr, self.info.size, float(mean), 0., 0., float(rtype(self.bias)),
                        stream_handle(self.stream))
        check(status, 'density contrast')
        self.mesh_delta = delta

    def _on_device(self, dtype):
        """Whether numpy's algebra of positions of ``dtype`` stays in that dtype, as the device's does."""
        if np.dtype(dtype) not in (np.dtype('f4'), np.dtype('f8')): return False
        return self._device_dtype(dtype) or (self.los is None and not self.wrap)

    @property
    def _positions_rec_data(self):
        """Reconstructed real-space positions of the data, on the host."""
        rec = self._rec_data
        return rec.numpy(stream=self.stream) if isinstance(rec, DeviceArray) else rec

    def run(self, niterations=3):
        """Reconstructed real-space data positions and the displacement meshes :attr:`mesh_psi`
        (iterative_fft_particle.py:61-78)."""
        if self.mesh_data.buffer is None or not hasattr(self, 'smoothing_radius'):
            raise ReconstructionError('assign data and set the density contrast before running')
        self._iter = 0
        self.mesh_data.smooth_gaussian(self.smoothing_radius)
        if self.has_randoms: self.mesh_randoms.smooth_gaussian(self.smoothing_radius)
        dtype = self._positions_data.dtype
        if self._on_device(dtype) and keeps_dtype(dtype, self.f, self.bias):
            self._data, _ = as_device(self._positions_data, stream=self.stream)
            self._rec_data = self._data
            self._data_weights, _ = as_device(self._weights_data, stream=self.stream)
        else:
            self._data = self._data_weights = None
            self._rec_data = self._positions_data.copy()
        for it in range(niterations):
            self.mesh_psi = self._iterate(return_psi=it == niterations - 1)
        self._data_weights = None
        self.mesh_randoms = None

    def _iterate(self, return_psi=False):
        """One iteration (iterative_fft_particle.py:80-139)."""
        self.logger.info('Running iteration {:d}.'.format(self._iter))
        if self._iter > 0:
            self.mesh_data = RealMesh(info=self.info, workspace=self.workspace, stream=self.stream)
            # paint the reconstructed real-space data positions, wrapped
            wrap = self.wrap
            self.wrap = True
            BaseReconstruction.assign_data(self, self._rec_data, weights=self._weights_data if self._data is None
                                           else self._data_weights)
            self.wrap = wrap
            self.mesh_data.smooth_gaussian(self.smoothing_radius)
        self.set_density_contrast(ran_min=self.ran_min, smoothing_radius=self.smoothing_radius)
        self.mesh_data = None
        # no displacement is needed along an axis the line of sight does not touch
        skipped = [not return_psi and self.los is not None and self.los[iaxis] == 0 for iaxis in range(3)]
        psis = self._compute_psi(skipped)
        self.mesh_delta = None
        first = self.beta / (1 + self.beta) if self._iter == 0 else 0.
        outside = False
        if self._data is not None:
            shifts = self._read_psi_device(self._rec_data, wrap=True, psis=psis)
            # the RSD is removed from the original positions; the next iteration paints these
            self._rec_data = self._point_algebra(_lib.POINT_ITERATE, self._data, s=shifts, first=first, out=shifts,
                                                 skip=sum(skip << iaxis for iaxis, skip in enumerate(skipped)),
                                                 outside=not self.wrap)
            if not self.wrap: self._rec_data, outside = self._rec_data
        else:
            shifts = np.zeros_like(self._rec_data)
            pos, _ = as_device(self._rec_data, stream=self.stream)
            for iaxis, psi in enumerate(psis):
                if not skipped[iaxis]: shifts[:, iaxis] = psi.read_cic(pos, wrap=True).numpy(stream=self.stream)
            if self.los is None:
                los = self._positions_data / distance(self._positions_data)[:, None]
            else:
                los = self.los
            if self._iter == 0:
                # first iteration: remove the RSD part approximately (Burden et al. 2015, eq. 12)
                shifts -= first * np.sum(shifts * los, axis=-1)[:, None] * los
            self._rec_data = self._positions_data - self.f * np.sum(shifts * los, axis=-1)[:, None] * los
            outside = self._out_of_bounds(self._rec_data)
        if outside: self.logger.warning('Some particles are out-of-bounds.')
        self._iter += 1
        if return_psi:
            return psis

    def _out_of_bounds(self, positions):
        diff = positions - self.info.offset
        return (not self.wrap) and np.any((diff < 0) | (diff > self.info.boxsize - self.info.cellsize))

    def _compute_psi(self, skipped):
        """The displacement meshes of :attr:`mesh_delta`; any mesh stands in for a skipped axis."""
        scratch = self._scratch(_lib.SPECTRAL_DISPLACEMENTS)
        if scratch is not None:
            return self._half_spectrum_psi(self.mesh_delta, scratch)
        delta_k = self._spectrum(self.mesh_delta)
        self._spectral(_lib.SPEC_INV_K2, delta_k, delta_k)
        work = self._complex()
        psis = [None] * 3
        for iaxis in range(3):
            if skipped[iaxis]: continue
            self._spectral(_lib.SPEC_I_KA, delta_k, work, a=iaxis, norm=1. / self.info.size)
            psis[iaxis] = self._to_real(work)
        done = next(psi for psi in psis if psi is not None)
        return [done if psi is None else psi for psi in psis]

    def _read_psi(self, positions, wrap=False):
        shifts = np.empty_like(positions)
        pos, _ = as_device(positions, stream=self.stream)
        for iaxis, psi in enumerate(self.mesh_psi):
            shifts[:, iaxis] = psi.read_cic(pos, wrap=wrap).numpy(stream=self.stream)
        return shifts

    def read_shifts(self, positions, field='disp+rsd'):
        """Displacements at ``positions``, or with ``positions='data'`` at the reconstructed data
        (iterative_fft_particle.py:141-212)."""
        return self._shifts(positions, self._check_field(field), False)

    def read_shifted_positions(self, positions, field='disp+rsd'):
        """``positions - read_shifts(positions)`` (``'data'``: the data given to :meth:`assign_data`), wrapped
        if :attr:`wrap` (iterative_fft_particle.py:214-239)."""
        if not isinstance(positions, str) and keeps_class(positions):
            positions = positions - self._shifts(positions, self._check_field(field), False)
            return self.info.wrap(positions) if self.wrap else positions
        return self._shifts(positions, self._check_field(field), True)

    def _shifts(self, positions, field, shifted):
        """Shifts or shifted positions (host arrays out)."""
        data = isinstance(positions, str) and positions == 'data'
        view = device_view(positions)
        if not data: positions = view if view is not None else np.asarray(positions)
        on_device = self._data is not None if data else \
            positions.ndim == 2 and positions.shape[1] == 3 and self._on_device(positions.dtype) \
            and (field == 'disp' or keeps_dtype(positions.dtype, self.f))
        if on_device and self._psi_on_mesh():
            return self._device_shifts(None if data else positions, field, shifted).numpy(stream=self.stream)
        if view is not None: positions = view.numpy(stream=self.stream)
        shifts = self._host_shifts(positions, field)
        if not shifted: return shifts
        positions = (self._positions_data if data else positions) - shifts
        if self.wrap: positions = self.info.wrap(positions)
        return positions

    def _device_shifts(self, positions, field, shifted):
        """On the device, as a device array; ``None`` stands for the data."""
        code = self._FIELDS[field]
        if positions is None:
            psi = self._read_psi_device(self._rec_data, wrap=True) if field != 'rsd' else self._rec_data
            return self._point_algebra(_lib.POINT_DATA, self._data, a=self._rec_data, s=psi, field=code, shifted=shifted)
        pos, _ = as_device(positions, stream=self.stream)
        inside = self._point_algebra(_lib.POINT_WRAP, pos) if self.wrap else pos
        psi = self._read_psi_device(inside)
        moved = None
        if field == 'disp+rsd':
            # the original algorithm's convention: RSD removed first, then the displacement read there
            real = self._point_algebra(_lib.POINT_REAL, inside, s=psi, outside=not self.wrap)
            if not self.wrap:
                real, outside = real
                if outside: self.logger.warning('Some particles are out-of-bounds.')
            moved = self._read_psi_device(real, wrap=True)
        return self._point_algebra(_lib.POINT_PARTICLE, inside, a=pos, s=psi, t=moved, field=code, shifted=shifted,
                                   out=psi)

    def _host_shifts(self, positions, field):
        """The shifts with the reference's numpy algebra on the host."""
        if isinstance(positions, str):
            positions = self._positions_rec_data
            shifts = self._read_psi(positions, wrap=True)
            if field == 'disp':
                return shifts
            rsd = self._positions_data - positions
            if field == 'rsd':
                return rsd
            shifts += rsd
            return shifts
        if self.wrap: positions = self.info.wrap(positions)
        shifts = self._read_psi(positions, wrap=False)
        if field == 'disp':
            return shifts
        if self.los is None:
            los = positions / distance(positions)[:, None]
        else:
            los = self.los
        rsd = self.f * np.sum(shifts * los, axis=-1)[:, None] * los
        if field == 'rsd':
            return rsd
        real_positions = positions - rsd
        if self._out_of_bounds(real_positions): self.logger.warning('Some particles are out-of-bounds.')
        shifts = self._read_psi(real_positions, wrap=True)
        return shifts + rsd


class IterativeFFTParticleReconstruction(OriginalIterativeFFTParticleReconstruction):
    """Any update upon the original algorithm (iterative_fft_particle.py:242-245)."""
