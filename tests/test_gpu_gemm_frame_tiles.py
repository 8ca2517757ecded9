"""Frame plans with their GEMMs on tiles other than the plan's own, through the
spec's gemm_config, against the oracle within the plan tolerance."""
import numpy as np
import pytest

from chestnut import Engine
from chestnut import spec as S
from chestnut import tune as TU
from oracle import model as OM
from test_gpu_engine import REL, frame_inputs, rel_err

pytestmark = pytest.mark.gpu


def frames_match(sp, cfg):
    """Two recurrent frames of the spec under a gemm_config, against the oracle."""
    w = S.make_weights(sp)
    orc = OM.OracleModel(sp, w, acc=np.float64)
    rng = np.random.default_rng(7)
    print(f'[frame] {sp["name"]} {cfg}', flush=True)
    with Engine(dict(sp, gemm_config=cfg), weights=w) as eng:
        hs = None
        for f, (warped, packed) in enumerate(frame_inputs(rng, sp['name'], 2)):
            if hs is not None:
                packed[12:] = hs
            out = eng.run_frame(warped, packed)
            ref = orc.run_frame(warped, packed)
            for name, sl in eng.out_slices.items():
                e = rel_err(out[sl], ref[sl])
                assert e <= REL, (f, name, e)
            hs = out[eng.out_slices['hidden_state']]


@pytest.mark.parametrize('spec', ['tiny', 'driving_39m'])
def test_every_gemm_at_tile_code_0(gpu, spec):
    """The automatic tile and split of every GEMM of the plan, the
    O-projection on a launch of its own among them."""
    sp = dict(S.get_spec(spec), n_layers=2, fuse_oproj=0)
    frames_match(sp, TU.config_for(sp, {fam: (0, 0) for fam in TU.shapes(sp)}))


@pytest.mark.parametrize('spec', ['tiny', 'driving_39m'])
@pytest.mark.parametrize('tile', [1, 9])
def test_qkv_on_128_and_256_row_tiles(gpu, spec, tile):
    """Two K-groups of 128x128 (tile 1) and 256x128 (tile 9), M below and at
    their rows."""
    sp = dict(S.get_spec(spec), n_layers=2)
    frames_match(sp, TU.config_for(sp, {'qkv': (tile, 1)}))


@pytest.mark.parametrize('spec,split', [('tiny', 1), ('tiny', 2), ('driving_39m', 4)])
@pytest.mark.parametrize('tile', [1, 9, 16])
def test_partials_and_embedding_on_the_pipelined_tiles(gpu, spec, split, tile):
    """The split-K partials that the next LayerNorm adds (O-projection, MLP
    down) and the embedding's epilogue on gemm_pipe_kernel."""
    sp = dict(S.get_spec(spec), n_layers=2, fuse_oproj=0)
    frames_match(sp, TU.config_for(sp, {'o': (tile, split), 'down': (tile, split), 'embed': (tile, 1)}))


@pytest.mark.parametrize('tile,split', [(1, 1), (9, 1), (16, 1), (17, 1), (9, 3), (16, 3)])
def test_batched_stem_on_the_pipelined_and_small_tiles(gpu, tile, split):
    """Two images per launch: stem layer 0, and the last layer, which the tiles
    without an implicit-conv A take through its patch matrix (K = 576)."""
    sp = dict(S.get_spec('tiny'), n_layers=2)
    cfg = {'stem0.conv': [tile, 1]}
    if tile != 1:
        cfg['stem4.conv'] = [tile, split]
    frames_match(sp, cfg)
