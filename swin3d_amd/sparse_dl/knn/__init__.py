from .knn import KNN, KNNInterpolate, KNNMaxPool, knn_interpolate, knn_max_pool, knn_query

__all__ = ["KNN", "KNNInterpolate", "KNNMaxPool", "knn_interpolate", "knn_max_pool", "knn_query"]
