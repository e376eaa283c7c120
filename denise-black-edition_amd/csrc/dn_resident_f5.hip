// Chip-resident time loop, FDORDER 10.
#define DN_F 5
#include "dn_resident_inst.inc"
