// Chip-resident time loop, FDORDER 6, acoustic, VTI, TTI and SH.
#define DN_F 3
#define DN_GROUP 1
#include "dn_resident_inst.inc"
