// Line lengths of the general pruned FFT, every sixth of the table (the files
// only divide the compile time).
#include "mn_fftg.h"

namespace mn {

const FgEntry *fg_entries_d(int *count) {
    static const FgEntry table[] = {
        fg::entry<9>(), fg::entry<20>(), fg::entry<36>(), fg::entry<60>(), fg::entry<90>(),
        fg::entry<128>(), fg::entry<180>(), fg::entry<243>(), fg::entry<320>(),
        fg::entry<405>(), fg::entry<512>(), fg::entry<648>(), fg::entry<800>(),
        fg::entry<1000>(), fg::entry<1215>(), fg::entry<1458>(), fg::entry<1800>(),
        fg::entry<2048>()};
    *count = (int)(sizeof(table) / sizeof(table[0]));
    return table;
}

}  // namespace mn
