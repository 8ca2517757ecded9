"""The GEMM planner (gemm_plan of gemm.hip) with every epilogue, called from a
small host program against the built library: tile code 0 for each GEMM of the
frame plans resolves to a tile that the epilogue runs on, and explicit tiles
stay what the caller named.  No GPU."""
import os
import subprocess

import pytest

from chestnut import _lib
from chestnut import spec as S
from chestnut import tune as TU
from conftest import PKG

HIPCC = os.environ.get('HIPCC', '/opt/rocm/bin/hipcc')
EPI = dict(f32=0, f16=1, relu=2, gelu=3, resid=4, qkv=5, partials=6, qkv_frag=7, embed=8)

PROGRAM = r'''
#include <cstdio>
#include <exception>
#include "kernels.h"
int main() {
  int M, N, K, batch, epi, conv_c, conv_h, conv_w, head_dim, tile, split;
  while (std::scanf("%d%d%d%d%d%d%d%d%d%d%d", &M, &N, &K, &batch, &epi, &conv_c, &conv_h, &conv_w, &head_dim, &tile,
                    &split) == 11) {
    ck::GemmDesc d;
    d.M = M; d.N = N; d.K = K; d.batch = batch; d.epi = epi;
    d.conv_c = conv_c; d.conv_h = conv_h; d.conv_w = conv_w;
    d.head_dim = head_dim;
    if (epi == ck::EPI_QKV || epi == ck::EPI_QKV_FRAG) d.qk_cols = N / 3 * 2;
    d.tile = tile; d.split = split;
    try {
      const size_t ws = ck::gemm_plan(d);
      std::printf("%d %d %zu\n", d.tile, d.split, ws);
    } catch (const std::exception& e) {
      std::printf("error %s\n", e.what());
    }
  }
}
'''


@pytest.fixture(scope='module')
def planner(tmp_path_factory):
    d = tmp_path_factory.mktemp('plan')
    (d / 'plan.cpp').write_text(PROGRAM)
    libdir = os.path.dirname(_lib.LIB_PATH)
    subprocess.run([HIPCC, '-std=c++17', '-O0', '--offload-arch=gfx950', '--offload-host-only',
                    '-I', os.path.join(PKG, 'csrc'), str(d / 'plan.cpp'), '-o', str(d / 'plan'), '-L', libdir,
                    '-lchestnut', f'-Wl,-rpath,{libdir}'], check=True, capture_output=True, text=True)

    def run(rows):
        text = '\n'.join(' '.join(str(v) for v in r) for r in rows) + '\n'
        out = subprocess.run([str(d / 'plan')], input=text, check=True, capture_output=True, text=True).stdout
        return [ln if ln.startswith('error') else tuple(int(v) for v in ln.split()) for ln in out.splitlines()]
    return run


def row(M, N, K, epi, batch=1, conv=(0, 0, 0), head_dim=0, tile=0, split=0):
    return (M, N, K, batch, EPI[epi], *conv, head_dim, tile, split)


def entries(sp):
    """name -> row of every GEMM of a spec's plan, at tile code 0."""
    out = {}
    H, W, C = sp['img_h'], sp['img_w'], 6 * sp['n_frames']
    for fam, (M, N, K, kind, batch) in TU.shapes(sp).items():
        if kind == 'conv':
            i = int(fam[4:])
            out[fam] = row(M, N, K, 'relu', batch, (sp['stem'][i - 1], sp['img_h'] >> i, sp['img_w'] >> i))
        else:
            epi = 'embed' if fam == 'embed' else {'frag': 'qkv_frag', 'partials': 'partials', 'f16': 'gelu',
                                                  'reduce': 'relu'}[kind]
            out[fam] = row(M, N, K, epi, batch, head_dim=sp['head_dim'])
    return out


@pytest.mark.parametrize('spec', ['tiny', 'driving_39m', 'big_driving_1b'])
@pytest.mark.parametrize('split', [0, 1])
def test_every_plan_entry_takes_tile_code_0(planner, spec, split):
    es = entries(S.get_spec(spec))
    got = planner([r[:-1] + (split,) for r in es.values()])
    assert len(got) == len(es)
    for (fam, r), g in zip(es.items(), got):
        assert not isinstance(g, str), (fam, g)
        if fam not in ('up', 'stem0'):   # what only the LDS-DMA tiles serve
            assert 1 <= g[0] <= 8, (fam, g)
        if split:
            assert g[1] == 1, (fam, g)


def test_tile_code_0_of_the_39m_entries(planner):
    es = entries(S.get_spec('driving_39m'))
    got = dict(zip(es, planner(list(es.values()))))
    assert got['qkv'][:2] == (4, 1) and got['o'][:2] == (4, 1) and got['down'][:2] == (4, 8)
    assert got['embed'][:2] == (4, 1) and got['stem3'][:2] == (4, 9) and got['stem4'][:2] == (4, 12)


@pytest.mark.parametrize('epi', ['f32', 'f16', 'relu', 'gelu', 'resid'])
def test_row_major_outputs_keep_the_small_and_large_tiles(planner, epi):
    got = planner([row(200, 520, 2048, epi), row(4096, 4096, 4096, epi), row(1000, 1000, 1024, epi)])
    assert [g[:2] for g in got] == [(17, 1), (9, 1), (16, 1)]


@pytest.mark.parametrize('epi', ['qkv', 'qkv_frag'])
def test_an_asked_qkv_tile_stays(planner, epi):
    """Tile 1 (two K-groups) and tile 9 (256x128) are kernels of their own for
    the QKV epilogues, not other names of tile 5."""
    tiles = [1, 2, 3, 4, 5, 8, 9, 15] + ([10] if epi == 'qkv_frag' else [])
    got = planner([row(512, 6144, 2048, epi, head_dim=128, tile=t, split=1) for t in tiles])
    assert [g[:2] for g in got] == [(t, 1) for t in tiles]
