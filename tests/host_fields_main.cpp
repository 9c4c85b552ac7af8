// Host check of fields_by_component() (st_device.h), built with one field-hook
// file: prints 1 or 0, whether the hooks are found to be the per-component
// form.
#include <stdio.h>

#include "../spin-tracking_amd/csrc/st_device.h"

int main() {
    printf("%d\n", st::fields_by_component() ? 1 : 0);
    return 0;
}
