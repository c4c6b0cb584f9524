"""The geometry's statement of which kernels run (it names them in timelines), against the library's
conditions."""


def _geometry(**kw):
    from adfwi_amd.propagator.acoustic_kernels import AcousticGeometry
    g = object.__new__(AcousticGeometry)      # the rule only, without a device
    g.fuse_steps, g.shots_per_block, g.adj_shots_per_block, g.row_unroll, g.tile_z = 1, 0, 0, 0, 0
    g.Z, g.pitch = 464, 1280
    for k, v in kw.items():
        setattr(g, k, v)
    return g


def test_acoustic_tiles_run_where_the_library_takes_them():
    assert _geometry().tiled
    for option in ("shots_per_block", "adj_shots_per_block", "row_unroll", "tile_z"):
        assert not _geometry(**{option: 4}).tiled
    assert not _geometry(fuse_steps=0).tiled
    assert not _geometry(pitch=1281).tiled
    assert _geometry(Z=8192, pitch=13056).tiled and not _geometry(Z=8192, pitch=13120).tiled   # five planes: 2 GiB
