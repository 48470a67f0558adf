"""GPU parity of lb_layer_rows (a SmolLM layer over batch x seq rows in seven launches) and lb_rms_rows, through
FrozenSmolLayer against its staged CPU reference: rel-L2 <= 1e-2 on outputs, keys and values (the decoder's bar)
at the edges of the 16-row tiles, for every weight format and correction rank class.
"""
import copy

import numpy as np
import pytest
import torch

import lowbit_hip
import smollm_random
from conftest import announce
from torch_npu_lowbit import QuantizedLinear, quantize_weight
from torch_npu_lowbit_correction import LowRankCorrection
from torch_npu_smollm import _ROWS_ORDER, _SHAPES, FrozenSmolLayer
from torch_npu_smollm_io import FrozenSmolIO

pytestmark = pytest.mark.gpu


# Deviations of the weights: small ones leave a row nearly its residual; PEAKED ones give attention over many keys a
# few large probabilities and more than half of the output.
PEAKED = {'self_attn.q_proj.weight': 0.07, 'self_attn.k_proj.weight': 0.07, 'self_attn.v_proj.weight': 0.08,
          'self_attn.o_proj.weight': 0.08}


def layer(mode, rank=0, capacity=160, protected=(), seed=3, deviations={}):
    g = torch.Generator().manual_seed(seed)
    weights = {n: (torch.randn(s, generator=g) * deviations.get(n, 0.02) if len(s) == 2 else 1 + 0.1 * torch.randn(s, generator=g)).half()
               for n, s in _SHAPES.items()}
    packed = corrections = None
    if rank:
        packed = {n: quantize_weight(w, format='int8') for n, w in weights.items() if w.ndim == 2}
        corrections = {n: LowRankCorrection(s, rank, (torch.randn(rank, s[1], generator=g) * 0.01).half().numpy().tobytes(),
                                            (torch.randn(s[0], rank, generator=g) * 0.01).half().numpy().tobytes())
                       for n, s in _SHAPES.items() if len(s) == 2 and n not in protected}
    return FrozenSmolLayer(smollm_random.config(10000.0, 1), weights, mode=mode, packed_weights=packed,
                           corrections=corrections, capacity=capacity, fp16_projections=protected)


def rel(got, want):
    want = want.double()
    return float((got.cpu().double() - want).norm() / want.norm())


CASES = [('w8a16', 32, 1, 1), ('w8a16', 32, 1, 16), ('w8a16', 8, 3, 17), ('w8a16', 4, 1, 33), ('w8a16', 0, 2, 64),
         ('w4a16', 0, 1, 15), ('w4a16', 0, 5, 31), ('nf4a16', 0, 1, 77), ('fp16', 0, 2, 130), ('fp16', 0, 1, 3),
         ('w8a16', 24, 8, 20), ('nf4a16', 0, 4, 120)]


@pytest.mark.parametrize('mode,rank,batch,seq', CASES)
def test_layer_rows_prefill_and_decode(device, mode, rank, batch, seq):
    """A prefill of seq rows, then three tokens: every row equals the CPU reference of the whole sequence, and a
    second continuation of the first snapshot gives the same bits (the snapshot was not changed)."""
    announce('layer rows', mode, rank, batch, seq)
    lay = layer(mode, rank)
    assert 'rows' in lay._dev(device)
    x = torch.randn(batch, seq + 3, 576, generator=torch.Generator().manual_seed(seq)).half()
    want, trace = lay.reference_cpu(x)
    with torch.no_grad():
        out, first = lay.prefill(x[:, :seq].to(device))
        assert rel(out, want[:, :seq]) <= 1e-2
        outs, cache = [], first
        for t in range(3):
            o, cache = lay.decode(x[:, seq + t:seq + t + 1].to(device), cache)
            outs.append(o)
        assert rel(torch.cat(outs, 1), want[:, seq:]) <= 1e-2
        assert rel(cache.keys[:, :, :seq + 3], trace['keys']) <= 1e-2 and rel(cache.values[:, :, :seq + 3], trace['values']) <= 1e-2
        assert not cache.keys[:, :, seq + 3:].any() and not cache.values[:, :, seq + 3:].any()
        again, _ = lay.decode(x[:, seq:seq + 1].to(device), first)
        assert torch.equal(again, outs[0])
        assert rel(lay(x.to(device)), want) <= 1e-2


@pytest.mark.parametrize('mode,rank,batch,seq', [('w8a16', 4, 1, 33), ('fp16', 0, 2, 130), ('w8a16', 32, 1, 257),
                                                 ('fp16', 0, 3, 288), ('w4a16', 0, 1, 513), ('nf4a16', 0, 2, 700),
                                                 ('w8a16', 8, 1, 1025), ('w8a16', 0, 1, 2016)])
def test_layer_rows_attention_of_few_large_weights(device, mode, rank, batch, seq):
    """Past 256 keys attention takes further rounds of score tiles, recomputed exponentials and reloaded values: whole
    prefills, the same rows in two calls (the second at a start of its own), and a decode at the last slot.  Without
    their last 32 keys the last rows would move by ten times the bar and more."""
    announce('layer rows long', mode, rank, batch, seq)
    lay = layer(mode, rank, capacity=2016, deviations=PEAKED)
    x = torch.randn(batch, seq, 576, generator=torch.Generator().manual_seed(seq)).half()
    want, trace = lay.reference_cpu(x)
    dev, rows = x.to(device), lay._dev(device)['rows']
    with torch.no_grad():
        out, cache = lay.prefill(dev)
        assert rel(out, want) <= 1e-2 and rel(out[:, -17:], want[:, -17:]) <= 1e-2
        assert rel(cache.keys[:, :, :seq], trace['keys']) <= 1e-2 and rel(cache.values[:, :, :seq], trace['values']) <= 1e-2
        keys, values = torch.zeros(2, batch, 3, 2016, 64, dtype=torch.float16, device=device)
        first = seq // 2 + 3
        parts = [rows.run(dev[:, :first], keys, values, 0), rows.run(dev[:, first:], keys, values, first)]
        assert rel(torch.cat(parts, 1), want) <= 1e-2 and rel(keys, cache.keys.cpu()) <= 1e-2
        _, short = lay.prefill(dev[:, :-1])
        last, _ = lay.decode(dev[:, -1:], short)
        assert rel(last, want[:, -1:]) <= 1e-2


def test_layer_rows_do_not_read_past_the_position(device):
    """Slots past the new token hold NaN and infinities; a strided input row is taken as it is."""
    announce('layer rows poison')
    lay = layer('w4a16')
    x = torch.randn(2, 40, 1152, generator=torch.Generator().manual_seed(1)).half()[..., ::2]
    with torch.no_grad():
        _, cache = lay.prefill(x[:, :35].to(device))
        want, _ = lay.decode(x[:, 35:36].to(device).clone(), cache)
        cache.keys[:, :, 36:] = float('nan')
        cache.values[:, :, 36:] = float('inf')
        got, _ = lay.decode(x.to(device)[:, 35:36], cache)
    assert torch.equal(got, want)


@pytest.mark.parametrize('protected,rows', [(('self_attn.o_proj.weight', 'mlp.down_proj.weight'), True),
                                            (('self_attn.q_proj.weight',), False)])
def test_layer_rows_and_protected_projections(device, protected, rows):
    """fp16-protected projections: in lb_layer_rows where q, k, v and gate, up keep one format, staged otherwise."""
    announce('layer rows protected', protected)
    lay = layer('w8a16', 32, protected=protected)
    assert ('rows' in lay._dev(device)) == rows
    x = torch.randn(1, 20, 576, generator=torch.Generator().manual_seed(2)).half()
    want, _ = lay.reference_cpu(x)
    with torch.no_grad():
        assert rel(lay(x.to(device)), want) <= 1e-2
        assert torch.equal(lay._full(x.to(device), None), lay.prefill(x.to(device))[0])   # forward keeps no cache


@pytest.mark.parametrize('rows,width', [(1, 576), (5, 8), (3, 4096), (257, 520)])
def test_rms_rows(device, rows, width):
    announce('rms rows', rows, width)
    g = torch.Generator().manual_seed(rows)
    x, gamma = torch.randn(rows, width, generator=g).half(), torch.randn(width, generator=g).half()
    f = x.float()
    want = (f * torch.rsqrt(f.square().mean(-1, keepdim=True) + 1e-5)).half() * gamma
    got = lowbit_hip.rms_rows(x.to(device), gamma.to(device)).cpu()
    # one fp16 rounding of the normalised value may fall on the other side of a tie, one of the product follows
    assert (np.abs(got.float().numpy() - want.float().numpy()) <= 2 ** -9 * np.abs(want.float().numpy()) + 2 ** -24).all()


def test_rows_at_any_address(device):
    """Contiguous views that begin at an odd element (2-byte aligned) give the bits of an aligned copy, through
    forward, prefill, decode and the logits, whose norm may be such a view too."""
    announce('rows at any address')
    lay = layer('w8a16', 8)
    g = torch.Generator().manual_seed(9)
    io = FrozenSmolIO(smollm_random.config(10000.0, 1), torch.randn(49152, 576, generator=g) * 0.02,
                      1 + 0.1 * torch.randn(576, generator=g)).to(device)
    for batch, seq in ((1, 1), (2, 5)):
        flat = torch.randn(batch * seq * 576 + 1, generator=g).half().to(device)
        odd = flat[1:].view(batch, seq, 576)
        x = odd.clone()
        assert odd.data_ptr() % 16 and odd.is_contiguous() and x.data_ptr() % 16 == 0
        with torch.no_grad():
            assert torch.equal(lay(odd), lay(x)) and torch.equal(io.logits(odd), io.logits(x))
            (a, cache), (b, _) = lay.prefill(odd), lay.prefill(x)
            assert torch.equal(a, b)
            assert torch.equal(lay.decode(odd[:, :1], cache)[0], lay.decode(x[:, :1].contiguous(), cache)[0])
    want = io.logits(x)
    io.norm = torch.cat((io.norm[:1], io.norm))[1:]
    assert io.norm.data_ptr() % 16 and torch.equal(io.logits(x), want)


def test_copies_of_used_modules(device):
    """Deep copies of a layer and a module that ran bind their own device state and give the same bits."""
    announce('copies')
    lay = layer('w8a16', 8)
    mod = QuantizedLinear(quantize_weight(torch.randn(64, 96) * 0.02, format='int4', group_size=32), bias=torch.randn(64))
    x, row = torch.randn(1, 5, 576).half().to(device), torch.randn(7, 192).half().to(device)[:, ::2]
    with torch.no_grad():
        for a, arg in ((lay, x), (mod, row)):
            want = a(arg)
            assert torch.equal(copy.deepcopy(a)(arg), want) and torch.equal(a(arg.contiguous()), want)


def test_padded_factors_are_complete_for_every_stream(device, monkeypatch):
    """Factors of odd ranks are padded on the stream of the first call, whose work the constructor waits for."""
    announce('padded factors')
    waited = []
    monkeypatch.setattr(torch.cuda.Stream, 'synchronize', lambda self: waited.append(torch.cuda.synchronize(device)))
    for rank, waits in ((8, 0), (4, 1)):
        waited.clear()
        lay = layer('w8a16', rank)
        lay._dev(device)
        assert len(waited) == waits
        x = torch.randn(1, 3, 576, generator=torch.Generator().manual_seed(8)).half()
        with torch.no_grad(), torch.cuda.stream(torch.cuda.Stream(device)):
            assert rel(lay(x.to(device)), lay.reference_cpu(x)[0]) <= 1e-2


def test_layer_rows_refuses(device):
    announce('layer rows refuses')
    lay = layer('w4a16', capacity=8)
    rows = lay._dev(device)['rows']
    x = torch.zeros(1, 4, 576, dtype=torch.float16, device=device)
    both = torch.zeros(2, 1, 3, 8, 64, dtype=torch.float16, device=device)
    for start in (-1, 5):
        with pytest.raises(ValueError, match='capacity'):
            rows.run(x, both[0], both[1], start)
    with pytest.raises(ValueError, match='overlaps'):
        rows.run(x, both[0], both[0], 0)


def test_one_row_over_a_long_cache(device):
    """A cache of 60000 slots, whose scores would not fit in LDS: one row at slot 10 gives the bits of a short cache."""
    announce('one row, long cache')
    outs = []
    for capacity in (16, 60000):
        lay = layer('w8a16', 8, capacity=capacity)
        state = lay._dev(device)
        rows = lowbit_hip.LayerRows([state['lin'][n] for n in _ROWS_ORDER], hidden=576, intermediate=1536,
                                    norm1=state['norm1'], norm2=state['norm2'], eps=1e-5, heads=9, kv_heads=3,
                                    cos=state['cos'], sin=state['sin'])
        x = torch.randn(1, 11, 576, generator=torch.Generator().manual_seed(6)).half().to(device)
        keys, values = torch.zeros(2, 1, 3, capacity, 64, dtype=torch.float16, device=device)
        rows.run(x[:, :10], keys, values, 0)
        outs.append((rows.run(x[:, 10:], keys, values, 10), keys[:, :, :16].clone(), values[:, :, :16].clone()))
    assert all(torch.equal(a, b) for a, b in zip(*outs))


def test_batches_past_the_launch_limits_are_staged(device):
    """65536 sequences (one past a grid's z range) still run, and 349184 rows within the limits: the last are a small batch's."""
    announce('layer rows limits')
    lay = layer('w4a16', capacity=8)
    rows = lay._dev(device)['rows']
    assert rows.fits(65535, 1) and rows.fits(1365, 256) and not rows.fits(65536, 1) and not rows.fits(1366, 256)
    x = torch.randn(64, 1, 576, generator=torch.Generator().manual_seed(4)).half().to(device)
    with torch.no_grad():
        want = lay(x)
        assert rel(lay(x.repeat(1024, 1, 1))[-64:], want.cpu()) <= 1e-2
        x = torch.randn(64, 8, 576, generator=torch.Generator().manual_seed(5)).half().to(device)
        assert rows.fits(64 * 682, 8) and not rows.fits(64 * 683, 8)
        want = lay(x)
        assert rel(lay(x.repeat(682, 1, 1))[-64:], want.cpu()) <= 1e-2   # 349184 rows in lb_layer_rows
