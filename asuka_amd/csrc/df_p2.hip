// Three-centre classes (32|c): instantiations of df_impl.h, compiled as a
// separate translation unit.
#include "df_impl.h"

#define ASUKA_DF_P2(X) X(3, 2, 0, 1) X(3, 2, 1, 3) X(3, 2, 2, 6) X(3, 2, 3, 10)

ASUKA_DF_FIND(find_df_p2, ASUKA_DF_P2)
