from .knn import KNN, KNNInterpolate, KNNInterpolateAdd, KNNMaxPool, interpolate_add_applies, knn_interpolate, knn_max_pool, knn_query

__all__ = ["KNN", "KNNInterpolate", "KNNInterpolateAdd", "KNNMaxPool", "interpolate_add_applies", "knn_interpolate", "knn_max_pool", "knn_query"]
