"""Host-side choice of the folded KV write (no GPU needed).

``forward_mixed`` and ``Attention.forward`` fold the store into the attention
launch only for new K/V rows stored back to back (``slo_attn.ops.foldable``),
and in decode steps also for views of a fused projection output
(``foldable_strided``); elsewhere such views keep the separate store launch.
"""
import torch

from slo_attn.ops import foldable, foldable_strided, folds_alone


def test_contiguous_rows_fold():
    k = torch.zeros(5, 8, 128, dtype=torch.bfloat16)
    assert foldable(k, k.clone())


def test_strided_views_and_other_dtypes_do_not_fold():
    qkv = torch.zeros(5, 48, 128, dtype=torch.bfloat16)  # q, k, v heads of a fused projection
    k, v = qkv[:, 32:40], qkv[:, 40:48]
    assert not foldable(k, v)
    kf = torch.zeros(5, 8, 128, dtype=torch.float32)
    assert not foldable(kf, kf.clone())
    kt = torch.zeros(5, 128, 8, dtype=torch.bfloat16).transpose(1, 2)  # heads not contiguous
    assert not foldable(kt, kt)


def test_decode_steps_fold_views_of_a_projection():
    qkv = torch.zeros(5, 48, 128, dtype=torch.bfloat16)
    k, v = qkv[:, 32:40], qkv[:, 40:48]
    assert foldable_strided(k, v) and foldable_strided(k.contiguous(), v)
    assert not foldable_strided(k.float(), v.float())
    assert not foldable_strided(k.expand(5, 8, 128).transpose(1, 2), v)  # heads not contiguous
    assert not foldable_strided(k[:1].expand(5, 8, 128), v)  # rows closer than a pool row
    odd = torch.zeros(5 * (1024 + 4), dtype=torch.bfloat16).as_strided((5, 8, 128), (1028, 128, 1))
    assert not foldable_strided(odd, v)  # rows off the 16-byte boundary


def test_steps_that_no_launch_carries_keep_the_store():
    qkv = torch.zeros(5, 48, 128, dtype=torch.bfloat16)
    q, k, v = qkv[:, :32], qkv[:, 32:40], qkv[:, 40:48]
    pool = torch.zeros(2, 64, 8, 128, dtype=torch.bfloat16)
    scale = torch.zeros(2, 64, 8)
    assert folds_alone(q, k, v, pool, None) and folds_alone(q, k, v, pool, scale)
    assert not folds_alone(q[:3], k, v, pool, None)  # more new rows than query rows
    assert not folds_alone(q, k[:3], v[:3], pool, scale)  # fewer
    assert not folds_alone(q, k, v, pool.view(2, 64, 1024), None)  # a pool view of merged heads
    wide = torch.zeros(5, 72, 128, dtype=torch.bfloat16)
    assert folds_alone(wide, k, v, pool, None) and not folds_alone(wide, k, v, pool, scale)  # 9 heads per kv head
