// Line lengths of the general pruned FFT, every sixth of the table (the files
// only divide the compile time).
#include "mn_fftg.h"

namespace mn {

const FgEntry *fg_entries_a(int *count) {
    static const FgEntry table[] = {
        fg::entry<4>(), fg::entry<15>(), fg::entry<27>(), fg::entry<48>(), fg::entry<75>(),
        fg::entry<108>(), fg::entry<150>(), fg::entry<216>(), fg::entry<270>(),
        fg::entry<375>(), fg::entry<480>(), fg::entry<600>(), fg::entry<729>(),
        fg::entry<900>(), fg::entry<1125>(), fg::entry<1296>(), fg::entry<1600>(),
        fg::entry<1944>()};
    *count = (int)(sizeof(table) / sizeof(table[0]));
    return table;
}

}  // namespace mn
