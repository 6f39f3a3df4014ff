// Adjoint and fused forward+adjoint kernel tables.  Generated by build.py.
#include "tri_adjoint.hpp"

namespace tri {

AdjTable<float> adj_table_f32() {
    static const AdjEntry<float> t[] = {
        {4, 8, 8, false, 0, 256, &launch_adj<float, 4, 8, 8, false, 0>},
        {8, 8, 8, false, 0, 512, &launch_adj<float, 8, 8, 8, false, 0>},
        {8, 8, 4, false, 0, 1024, &launch_adj<float, 8, 8, 4, false, 0>},
        {8, 8, 2, false, 0, 2048, &launch_adj<float, 8, 8, 2, false, 0>},
        {8, 8, 1, false, 0, 4096, &launch_adj<float, 8, 8, 1, false, 0>},
        {12, 8, 8, false, 0, 768, &launch_adj<float, 12, 8, 8, false, 0>},
        {12, 8, 4, false, 0, 1536, &launch_adj<float, 12, 8, 4, false, 0>},
        {12, 8, 2, false, 0, 3072, &launch_adj<float, 12, 8, 2, false, 0>},
        {12, 8, 1, false, 0, 6144, &launch_adj<float, 12, 8, 1, false, 0>},
        {8, 16, 1, false, 0, 8192, &launch_adj<float, 8, 16, 1, false, 0>},
        {4, 8, 8, false, 1, 256, &launch_adj<float, 4, 8, 8, false, 1>},
        {8, 8, 8, false, 1, 512, &launch_adj<float, 8, 8, 8, false, 1>},
        {8, 8, 4, false, 1, 1024, &launch_adj<float, 8, 8, 4, false, 1>},
        {8, 8, 2, false, 1, 2048, &launch_adj<float, 8, 8, 2, false, 1>},
        {8, 8, 1, false, 1, 4096, &launch_adj<float, 8, 8, 1, false, 1>},
        {12, 4, 4, false, 1, 768, &launch_adj<float, 12, 4, 4, false, 1>},
        {12, 4, 2, false, 1, 1536, &launch_adj<float, 12, 4, 2, false, 1>},
        {12, 4, 1, false, 1, 3072, &launch_adj<float, 12, 4, 1, false, 1>},
        {12, 8, 1, false, 1, 6144, &launch_adj<float, 12, 8, 1, false, 1>},
        {8, 16, 1, false, 1, 8192, &launch_adj<float, 8, 16, 1, false, 1>},
        {4, 1, 8, true, 0, 32, &launch_adj<float, 4, 1, 8, true, 0>},
        {4, 1, 8, true, 1, 32, &launch_adj<float, 4, 1, 8, true, 1>},
        {4, 2, 8, true, 0, 64, &launch_adj<float, 4, 2, 8, true, 0>},
        {4, 2, 8, true, 1, 64, &launch_adj<float, 4, 2, 8, true, 1>},
        {4, 4, 8, true, 0, 128, &launch_adj<float, 4, 4, 8, true, 0>},
        {4, 4, 8, true, 1, 128, &launch_adj<float, 4, 4, 8, true, 1>},
        {4, 8, 8, true, 0, 256, &launch_adj<float, 4, 8, 8, true, 0>},
        {4, 8, 8, true, 1, 256, &launch_adj<float, 4, 8, 8, true, 1>},
        {4, 16, 8, true, 0, 512, &launch_adj<float, 4, 16, 8, true, 0>},
        {4, 16, 8, true, 1, 512, &launch_adj<float, 4, 16, 8, true, 1>},
        {8, 1, 8, true, 0, 64, &launch_adj<float, 8, 1, 8, true, 0>},
        {8, 1, 8, true, 1, 64, &launch_adj<float, 8, 1, 8, true, 1>},
        {8, 2, 8, true, 0, 128, &launch_adj<float, 8, 2, 8, true, 0>},
        {8, 2, 8, true, 1, 128, &launch_adj<float, 8, 2, 8, true, 1>},
        {8, 4, 8, true, 0, 256, &launch_adj<float, 8, 4, 8, true, 0>},
        {8, 4, 8, true, 1, 256, &launch_adj<float, 8, 4, 8, true, 1>},
        {8, 8, 8, true, 0, 512, &launch_adj<float, 8, 8, 8, true, 0>},
        {8, 8, 8, true, 1, 512, &launch_adj<float, 8, 8, 8, true, 1>},
        {8, 16, 8, true, 0, 1024, &launch_adj<float, 8, 16, 8, true, 0>},
        {8, 16, 8, true, 1, 1024, &launch_adj<float, 8, 16, 8, true, 1>},
    };
    return {t, (int)(sizeof(t) / sizeof(t[0]))};
}

AdjTable<double> adj_table_f64() {
    static const AdjEntry<double> t[] = {
        {4, 8, 8, false, 0, 256, &launch_adj<double, 4, 8, 8, false, 0>},
        {6, 8, 8, false, 0, 384, &launch_adj<double, 6, 8, 8, false, 0>},
        {8, 8, 8, false, 0, 512, &launch_adj<double, 8, 8, 8, false, 0>},
        {8, 8, 4, false, 0, 1024, &launch_adj<double, 8, 8, 4, false, 0>},
        {8, 8, 2, false, 0, 2048, &launch_adj<double, 8, 8, 2, false, 0>},
        {8, 8, 1, false, 0, 4096, &launch_adj<double, 8, 8, 1, false, 0>},
        {12, 4, 4, false, 0, 768, &launch_adj<double, 12, 4, 4, false, 0>},
        {12, 4, 2, false, 0, 1536, &launch_adj<double, 12, 4, 2, false, 0>},
        {12, 4, 1, false, 0, 3072, &launch_adj<double, 12, 4, 1, false, 0>},
        {12, 8, 1, false, 0, 6144, &launch_adj<double, 12, 8, 1, false, 0>},
        {4, 8, 8, false, 1, 256, &launch_adj<double, 4, 8, 8, false, 1>},
        {6, 8, 8, false, 1, 384, &launch_adj<double, 6, 8, 8, false, 1>},
        {8, 4, 4, false, 1, 512, &launch_adj<double, 8, 4, 4, false, 1>},
        {8, 4, 2, false, 1, 1024, &launch_adj<double, 8, 4, 2, false, 1>},
        {8, 4, 1, false, 1, 2048, &launch_adj<double, 8, 4, 1, false, 1>},
        {12, 4, 4, false, 1, 768, &launch_adj<double, 12, 4, 4, false, 1>},
        {12, 4, 2, false, 1, 1536, &launch_adj<double, 12, 4, 2, false, 1>},
        {12, 4, 1, false, 1, 3072, &launch_adj<double, 12, 4, 1, false, 1>},
        {8, 8, 1, false, 1, 4096, &launch_adj<double, 8, 8, 1, false, 1>},
        {12, 8, 1, false, 1, 6144, &launch_adj<double, 12, 8, 1, false, 1>},
        {4, 1, 4, true, 0, 64, &launch_adj<double, 4, 1, 4, true, 0>},
        {4, 1, 4, true, 1, 64, &launch_adj<double, 4, 1, 4, true, 1>},
        {4, 2, 4, true, 0, 128, &launch_adj<double, 4, 2, 4, true, 0>},
        {4, 2, 4, true, 1, 128, &launch_adj<double, 4, 2, 4, true, 1>},
        {4, 4, 4, true, 0, 256, &launch_adj<double, 4, 4, 4, true, 0>},
        {4, 4, 4, true, 1, 256, &launch_adj<double, 4, 4, 4, true, 1>},
        {4, 8, 4, true, 0, 512, &launch_adj<double, 4, 8, 4, true, 0>},
        {4, 8, 4, true, 1, 512, &launch_adj<double, 4, 8, 4, true, 1>},
        {8, 1, 4, true, 0, 128, &launch_adj<double, 8, 1, 4, true, 0>},
        {8, 1, 4, true, 1, 128, &launch_adj<double, 8, 1, 4, true, 1>},
        {8, 2, 4, true, 0, 256, &launch_adj<double, 8, 2, 4, true, 0>},
        {8, 2, 4, true, 1, 256, &launch_adj<double, 8, 2, 4, true, 1>},
        {8, 4, 4, true, 0, 512, &launch_adj<double, 8, 4, 4, true, 0>},
        {8, 4, 4, true, 1, 512, &launch_adj<double, 8, 4, 4, true, 1>},
        {8, 8, 4, true, 0, 1024, &launch_adj<double, 8, 8, 4, true, 0>},
        {8, 8, 4, true, 1, 1024, &launch_adj<double, 8, 8, 4, true, 1>},
    };
    return {t, (int)(sizeof(t) / sizeof(t[0]))};
}

}  // namespace tri
